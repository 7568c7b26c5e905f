// Join driver: probe layer P against build layer R's LBVH (reference: join_stream, engine/engine.cuh:895-1061).
//
// Per probe batch (<= batch_q probes, a subdivided parent's pieces never split across batches): count pass, scan,
// write pass, refinement, compaction, piece -> parent aggregation, DE-9IM codes; then either a device-side consumer
// (cluster) or one copy of the rows into pinned host memory and the row callback.
//
// Compaction is split by what a candidate needs: a pair whose two parents are single pieces maps to its parent pair
// directly (kept iff its flag is 1). Only pairs touching a subdivided parent are sorted and folded, first by piece
// pair and then (stable) by parent pair, so every parent's terms are added in the same order as in the CPU
// restatement: a subdivided layer's aggregated areas are bit-identical too.
#include "scan.h"
#include <algorithm>
#include <chrono>

namespace gsj {

namespace {

__device__ __forceinline__ uint32_t parent_of(const DPolys& S, uint32_t g) { return S.parent ? S.parent[g] : g; }
__device__ __forceinline__ bool multi_piece(const DPolys& S, uint32_t p) { return S.pfirst && (S.pfirst[p + 1] - S.pfirst[p] > 1); }

// Kept candidates of layers without parents: flag 1, or any flag (no aggregation: piece pairs)
struct LoadHit {
  static constexpr bool PACKED = false;
  const uint8_t* f;
  int any;
  __device__ __forceinline__ bool keep(uint64_t i) const { return any ? f[i] != 0 : f[i] == 1; }
  __device__ __forceinline__ uint64_t operator()(uint64_t i) const { return keep(i) ? 1u : 0u; }
};
// Kept candidates of subdivided layers by what they need: low half single-piece rows (flag 1), high half candidates of a
// parent of several pieces (any flag), which go to the fold. One scan counts both.
constexpr uint8_t KIND_ROW = 1, KIND_FOLD = 2;
struct LoadKind {
  static constexpr bool PACKED = true;
  const uint8_t* kind;
  __device__ __forceinline__ uint64_t operator()(uint64_t i) const {
    const uint8_t k = kind[i];
    return k == KIND_ROW ? 1ull : k == KIND_FOLD ? 1ull << 32 : 0ull;
  }
};
__global__ void k_row_kinds(const DPolys P, const DPolys R, const uint32_t* __restrict__ pa, const uint32_t* __restrict__ pb,
                            const uint8_t* __restrict__ isect, uint64_t n, uint8_t* __restrict__ kind) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint8_t f = isect[i];
  uint8_t k = 0;
  if (f) {
    const bool multi = multi_piece(P, parent_of(P, pa[i])) || multi_piece(R, parent_of(R, pb[i]));
    k = multi ? KIND_FOLD : (f == 1 ? KIND_ROW : 0);
  }
  kind[i] = k;
}

__device__ __forceinline__ void put_row(const DPolys& P, const DPolys& R, uint32_t a, uint32_t b, uint32_t qa, uint32_t qb, uint64_t o, uint64_t i,
                                        const double* area, const double4* ev, const uint32_t* evb, uint32_t* orow, double* oarea, uint32_t* ocode) {
  reinterpret_cast<uint2*>(orow)[o] = make_uint2(a, b);
  if (oarea) oarea[o] = area[i];
  if (ocode) {
    const double4 e = ev[i];
    ocode[o] = de9im_code(e.x, e.y, e.z, e.w, evb[i], P.blen[qa], R.blen[qb]);
  }
}
__global__ void k_emit_hits(const DPolys P, const DPolys R, const uint32_t* __restrict__ pa, const uint32_t* __restrict__ pb, const LoadHit hit,
                            const uint64_t* __restrict__ offs, uint64_t n, const double* __restrict__ area, const double4* __restrict__ ev,
                            const uint32_t* __restrict__ evb, uint32_t* __restrict__ orow, double* __restrict__ oarea, uint32_t* __restrict__ ocode) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !hit.keep(i)) return;
  const uint32_t a = pa[i], b = pb[i];
  put_row(P, R, a, b, parent_of(P, a), parent_of(R, b), offs[i], i, area, ev, evb, orow, oarea, ocode);
}

// A folded candidate's place: parent pair, then piece pair. parent A | parent B | piece of A | piece of B within their
// parents, in the bits that the layers need (their pieces are numbered parent by parent). Where those exceed 63, `wide`:
// the piece pair first, and the parent pair as a second key (b = 32, la = lb = 0).
struct FoldKey {
  int b, la, lb;   // bits of parent B, of a piece of A, of a piece of B
  int wide;
  __device__ __forceinline__ uint64_t of(const DPolys& P, const DPolys& R, uint32_t ga, uint32_t gb) const {
    if (wide) return ((uint64_t)ga << 32) | gb;
    const uint32_t qa = parent_of(P, ga), qb = parent_of(R, gb);
    const uint64_t ia = P.pfirst ? ga - P.pfirst[qa] : 0u, ib = R.pfirst ? gb - R.pfirst[qb] : 0u;
    return ((((((uint64_t)qa << b) | qb) << la) | ia) << lb) | ib;
  }
  __device__ __forceinline__ uint64_t pair(uint64_t key) const { return key >> (la + lb); }
  __device__ __forceinline__ uint32_t row_a(uint64_t pair) const { return (uint32_t)(pair >> b); }
  __device__ __forceinline__ uint32_t row_b(uint64_t pair) const { return (uint32_t)(pair & ((1ull << b) - 1)); }
};

// single-piece rows to their places, folded candidates with their keys into the fold's list
__global__ void k_emit_kinds(const DPolys P, const DPolys R, const uint32_t* __restrict__ pa, const uint32_t* __restrict__ pb,
                             const uint8_t* __restrict__ kind, const uint64_t* __restrict__ offs, uint64_t n, const double* __restrict__ area,
                             const double4* __restrict__ ev, const uint32_t* __restrict__ evb, uint32_t* __restrict__ orow, double* __restrict__ oarea,
                             uint32_t* __restrict__ ocode, const FoldKey fk, uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint8_t k = kind[i];
  if (!k) return;
  const uint64_t o = offs[i];
  const uint32_t a = pa[i], b = pb[i];
  if (k == KIND_ROW) {
    const uint32_t qa = parent_of(P, a), qb = parent_of(R, b);
    put_row(P, R, qa, qb, qa, qb, o & 0xFFFFFFFFull, i, area, ev, evb, orow, oarea, ocode);
  } else {
    keys[o >> 32] = fk.of(P, R, a, b);
    vals[o >> 32] = (uint32_t)i;
  }
}

// the sum of a parent pair's piece pairs [j, end) in key order; whether it is a row (every piece pair's flag is 1)
struct FoldSum {
  double ar = 0, e0 = 0, e1 = 0, e2 = 0, e3 = 0;
  uint32_t bits = 0;
  uint8_t f = 255;
  __device__ __forceinline__ void add(uint32_t i, const uint8_t* isect, const double* area, const double4* ev, const uint32_t* evb) {
    if (area) ar += area[i];
    if (ev) { const double4 e = ev[i]; e0 += e.x; e1 += e.y; e2 += e.z; e3 += e.w; bits |= evb[i]; }
    f = min(f, isect[i]);
  }
};

// The whole fold of at most FOLD_MAX candidates in one block: a bitonic sort of (key, candidate) in LDS, then 1024
// positions at a time the parent pairs that start there are summed, the kept ones counted by ballot and written behind
// the single-piece rows. A subdivided layer has few parents of several pieces (parcels over 256 vertices: 1 in 5000), so
// nearly every request stays here: one launch instead of two radix sorts and four scans (some 100 launches and 5 waits;
// 51k parcels, self relate: 1.14 -> 0.79 ms). counts: single-piece rows | folded candidates << 32; out[0] = its rows.
constexpr uint32_t FOLD_MAX = 4096, FOLD_T = 1024;
__global__ void __launch_bounds__(FOLD_T) k_fold_small(const DPolys P, const DPolys R, const uint64_t* __restrict__ counts, const FoldKey fk,
                                                       const uint64_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                       const uint8_t* __restrict__ isect, const double* __restrict__ area,
                                                       const double4* __restrict__ ev, const uint32_t* __restrict__ evb, uint32_t* __restrict__ orow,
                                                       double* __restrict__ oarea, uint32_t* __restrict__ ocode, uint64_t* __restrict__ out) {
  __shared__ uint64_t K[FOLD_MAX];
  __shared__ uint32_t V[FOLD_MAX];
  __shared__ uint32_t wsum[FOLD_T / 64];
  const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
  const uint32_t m = (uint32_t)min(counts[0] >> 32, (uint64_t)0xFFFFFFFFull), nsingle = (uint32_t)counts[0];
  if (m == 0 || m > FOLD_MAX) {   // (more: the host sorts them)
    if (t == 0) out[0] = 0;
    return;
  }
  uint32_t N = 64;
  while (N < m) N <<= 1;
  for (uint32_t j = t; j < N; j += FOLD_T) {
    K[j] = j < m ? keys[j] : ~0ull;   // above every key (FOLD_KEY_BITS)
    V[j] = j < m ? vals[j] : 0u;
  }
  __syncthreads();
  for (uint32_t k = 2; k <= N; k <<= 1)
    for (uint32_t d = k >> 1; d > 0; d >>= 1) {
      for (uint32_t p = t; p < N / 2; p += FOLD_T) {
        const uint32_t i = (p & ~(d - 1)) * 2 + (p & (d - 1)), j = i + d;   // the p-th pair at distance d
        const uint64_t a = K[i], b = K[j];
        if ((a > b) == ((i & k) == 0)) {
          K[i] = b; K[j] = a;
          const uint32_t v = V[i];
          V[i] = V[j]; V[j] = v;
        }
      }
      __syncthreads();
    }
  uint32_t base = 0;
  for (uint32_t r = 0; r < m; r += FOLD_T) {
    const uint32_t j = r + t;
    bool keep = false;
    uint64_t pr = 0;
    FoldSum s;
    if (j < m) {
      pr = fk.pair(K[j]);
      if (j == 0 || fk.pair(K[j - 1]) != pr) {
        for (uint32_t q = j; q < m && fk.pair(K[q]) == pr; q++) s.add(V[q], isect, area, ev, evb);
        keep = s.f == 1;
      }
    }
    const uint64_t bal = __ballot(keep);
    if (lane == 0) wsum[w] = (uint32_t)__popcll(bal);
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t q = 0; q < FOLD_T / 64; q++) {
      if (q < w) before += wsum[q];
      all += wsum[q];
    }
    if (keep) {
      const uint32_t o = nsingle + base + before + (uint32_t)__popcll(bal & ((1ull << lane) - 1));
      const uint32_t qa = fk.row_a(pr), qb = fk.row_b(pr);
      reinterpret_cast<uint2*>(orow)[o] = make_uint2(qa, qb);
      if (oarea) oarea[o] = s.ar;
      if (ocode) ocode[o] = de9im_code(s.e0, s.e1, s.e2, s.e3, s.bits, P.blen[qa], R.blen[qb]);
    }
    base += all;
    __syncthreads();   // wsum is rewritten
  }
  if (t == 0) out[0] = base;
}

// the second key of the folded candidates
__global__ void k_parent_keys(const DPolys P, const DPolys R, const uint32_t* __restrict__ pa, const uint32_t* __restrict__ pb,
                              const uint32_t* __restrict__ vals, uint64_t m, uint64_t* __restrict__ keys) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= m) return;
  const uint32_t i = vals[j];
  keys[j] = ((uint64_t)parent_of(P, pa[i]) << 32) | parent_of(R, pb[i]);
}

__global__ void k_heads(const uint64_t* __restrict__ keys, uint64_t m, const FoldKey fk, uint32_t* __restrict__ head) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < m) head[j] = (j == 0 || fk.pair(keys[j]) != fk.pair(keys[j - 1])) ? 1u : 0u;
}

__global__ void k_seg_starts(const uint32_t* __restrict__ head, const uint64_t* __restrict__ hoff, uint64_t m, uint64_t* __restrict__ start) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < m && head[j]) start[hoff[j]] = j;
}

// one thread per parent pair: terms added in (piece a, piece b) order; flag = min over its piece pairs
__global__ void k_seg_fold(const uint32_t* __restrict__ vals, const uint64_t* __restrict__ start, uint64_t nseg, uint64_t m,
                           const uint8_t* __restrict__ isect, const double* __restrict__ area, const double4* __restrict__ ev,
                           const uint32_t* __restrict__ evb, uint32_t* __restrict__ keep, double* __restrict__ sarea, double4* __restrict__ sev,
                           uint32_t* __restrict__ sevb) {
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  const uint64_t j0 = start[s], j1 = s + 1 < nseg ? start[s + 1] : m;
  FoldSum f;
  for (uint64_t j = j0; j < j1; j++) f.add(vals[j], isect, area, ev, evb);
  keep[s] = f.f == 1;
  sarea[s] = f.ar;
  if (ev) { sev[s] = make_double4(f.e0, f.e1, f.e2, f.e3); sevb[s] = f.bits; }
}

__global__ void k_emit_multi(const DPolys P, const DPolys R, const uint64_t* __restrict__ keys, const FoldKey fk, const uint64_t* __restrict__ start,
                             const uint32_t* __restrict__ keep, const uint64_t* __restrict__ koff, uint64_t nseg, uint64_t base,
                             const double* __restrict__ sarea, const double4* __restrict__ sev, const uint32_t* __restrict__ sevb,
                             uint32_t* __restrict__ orow, double* __restrict__ oarea, uint32_t* __restrict__ ocode) {
  const uint64_t s = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg || !keep[s]) return;
  const uint64_t o = base + koff[s];
  const uint64_t k = fk.pair(keys[start[s]]);
  const uint32_t a = fk.row_a(k), b = fk.row_b(k);
  orow[2 * o] = a; orow[2 * o + 1] = b;
  if (oarea) oarea[o] = sarea[s];
  if (ocode) { const double4 e = sev[s]; ocode[o] = de9im_code(e.x, e.y, e.z, e.w, sevb[s], P.blen[a], R.blen[b]); }
}

inline int bits_for(uint64_t maxval) { int b = 1; while (b < 64 && (maxval >> b)) b++; return b; }

}  // namespace

namespace {

constexpr int FOLD_KEY_BITS = 63;   // a packed fold key's bits: 64 ones are the block sort's padding, which has to come last

// Compaction of one sub-batch's refined candidates into parent-pair rows at (orow, oarea, ocode: device memory, or pinned
// host memory that the kernels write directly). compact_enqueue asks for no host wait; after the caller's, the row
// count comes from compact_finish, which folds here only what did not fit one block.
struct Compaction {
  const Layer* PL;
  const Layer* RL;
  const uint32_t* pa;
  const uint32_t* pb;
  uint64_t np;
  RefineParams rp;
  RefineOut ro;
  uint32_t* orow;
  double* oarea;     // null when not asked for
  uint32_t* ocode;
  bool fold;         // some parent has several pieces
  FoldKey fk;
  int key_bits;
  const uint64_t* offs;   // of the kept candidates (without fold)
  HostWords words;        // [0] single-piece rows | folded candidates << 32, [1] rows folded in one block
  bool host_folds() const { return fold && (fk.wide || (words.host[0] >> 32) > FOLD_MAX); }   // (after the wait)
};

Compaction compact_enqueue(Context& c, const Layer& PL, const Layer& RL, const uint32_t* pa, const uint32_t* pb, uint64_t np, const RefineParams& rp,
                           const RefineOut& ro, bool no_agg, uint32_t* orow, double* oarea, uint32_t* ocode) {
  hipStream_t st = c.stream;
  const DPolys& P = PL.poly;
  const DPolys& R = RL.poly;
  Compaction k{&PL, &RL, pa, pb, np, rp, ro, orow, rp.want_area ? oarea : nullptr, rp.want_relate ? ocode : nullptr, !no_agg && (P.pfirst || R.pfirst),
               FoldKey{}, 0, nullptr, host_words(c, 0, 2)};
  uint64_t* offs = c.s_offs.as<uint64_t>(np + 16);
  k.offs = offs;
  if (!k.fold) {
    const LoadHit hit{ro.isect, no_agg ? 1 : 0};
    scan_loaded<uint64_t>(c, hit, offs, np, ScanTotal{k.words.dev});
    hipLaunchKernelGGL(k_emit_hits, dim3(div_up(np, 256)), dim3(256), 0, st, P, R, pa, pb, hit, offs, np, ro.area, ro.ev, ro.evb, orow, k.oarea, k.ocode);
    GSJ_LAUNCHED();
    return k;
  }
  k.fk = FoldKey{bits_for(std::max<uint64_t>(RL.nparent, 1) - 1), bits_for(PL.max_pieces - 1), bits_for(RL.max_pieces - 1), 0};
  k.key_bits = bits_for(std::max<uint64_t>(PL.nparent, 1) - 1) + k.fk.b + k.fk.la + k.fk.lb;
  if (k.key_bits > FOLD_KEY_BITS) k.fk = FoldKey{32, 0, 0, 1};
  uint8_t* kind = c.s_tmp.as<uint8_t>(np + 16);
  uint64_t* dtotal = c.s_words.as<uint64_t>(HOST_WORDS) + 16;
  uint64_t* keys = c.s_keys.as<uint64_t>(np + 16);
  uint32_t* vals = c.s_vals.as<uint32_t>(np + 16);
  hipLaunchKernelGGL(k_row_kinds, dim3(div_up(np, 256)), dim3(256), 0, st, P, R, pa, pb, ro.isect, np, kind);
  GSJ_LAUNCHED();
  scan_loaded<uint64_t>(c, LoadKind{kind}, offs, np, ScanTotal{k.words.dev, nullptr, dtotal});
  hipLaunchKernelGGL(k_emit_kinds, dim3(div_up(np, 256)), dim3(256), 0, st, P, R, pa, pb, kind, offs, np, ro.area, ro.ev, ro.evb, orow, k.oarea, k.ocode,
                     k.fk, keys, vals);
  GSJ_LAUNCHED();
  const bool rel = rp.want_relate != 0;
  if (k.fk.wide) return k;   // the host sorts them
  hipLaunchKernelGGL(k_fold_small, dim3(1), dim3(FOLD_T), 0, st, P, R, dtotal, k.fk, keys, vals, ro.isect, rp.want_area ? ro.area : nullptr,
                     rel ? ro.ev : nullptr, rel ? ro.evb : nullptr, orow, k.oarea, k.ocode, k.words.dev + 1);
  GSJ_LAUNCHED();
  return k;
}

uint64_t compact_finish(Context& c, const Compaction& k) {
  const uint64_t total = k.words.host[0];
  if (!k.fold) return total;
  const uint64_t nsingle = total & 0xFFFFFFFFull, m = total >> 32;
  if (!k.host_folds()) return nsingle + (m ? k.words.host[1] : 0);
  if (m == 0) return nsingle;
  hipStream_t st = c.stream;
  const DPolys& P = k.PL->poly;
  const DPolys& R = k.RL->poly;
  uint64_t* keys = c.s_keys.as<uint64_t>(k.np + 16);
  uint64_t* keys2 = c.s_keys2.as<uint64_t>(k.np + 16);
  uint32_t* vals = c.s_vals.as<uint32_t>(k.np + 16);
  uint32_t* vals2 = c.s_vals2.as<uint32_t>(k.np + 16);
  radix_sort_pairs(c, keys, keys2, vals, vals2, m, 0, k.fk.wide ? 64 : k.key_bits);
  if (k.fk.wide) {   // piece-pair order, then stable parent-pair order
    hipLaunchKernelGGL(k_parent_keys, dim3(div_up(m, 256)), dim3(256), 0, st, P, R, k.pa, k.pb, vals, m, keys);
    GSJ_LAUNCHED();
    radix_sort_pairs(c, keys, keys2, vals, vals2, m, 0, 32 + bits_for(std::max<uint64_t>(k.PL->nparent, 1)));
  }
  uint32_t* head = c.s_seg.as<uint32_t>(3 * m + 16);
  uint32_t* keep = head + m;
  uint64_t* hoff = c.s_tmp2.as<uint64_t>(2 * m + 16);
  hipLaunchKernelGGL(k_heads, dim3(div_up(m, 256)), dim3(256), 0, st, keys, m, k.fk, head);
  GSJ_LAUNCHED();
  const uint64_t nseg = scan_u32_to_u64(c, head, hoff, m);
  uint64_t* start = hoff + m;
  hipLaunchKernelGGL(k_seg_starts, dim3(div_up(m, 256)), dim3(256), 0, st, head, hoff, m, start);
  GSJ_LAUNCHED();
  double* sarea = c.s_out_flag.as<double>(nseg * 6 + 16);
  double4* sev = reinterpret_cast<double4*>(sarea + ((nseg + 3) & ~uint64_t(3)));
  uint32_t* sevb = reinterpret_cast<uint32_t*>(sev + nseg);
  const bool rel = k.rp.want_relate != 0;
  hipLaunchKernelGGL(k_seg_fold, dim3(div_up(nseg, 256)), dim3(256), 0, st, vals, start, nseg, m, k.ro.isect, k.rp.want_area ? k.ro.area : nullptr,
                     rel ? k.ro.ev : nullptr, rel ? k.ro.evb : nullptr, keep, sarea, sev, sevb);
  GSJ_LAUNCHED();
  uint64_t* koff = c.s_offs.as<uint64_t>(std::max<uint64_t>(k.np, nseg) + 16);   // the candidates' offsets are no longer needed
  const uint64_t nkeep = scan_u32_to_u64(c, keep, koff, nseg);
  hipLaunchKernelGGL(k_emit_multi, dim3(div_up(nseg, 256)), dim3(256), 0, st, P, R, keys, k.fk, start, keep, koff, nseg, nsingle, sarea, sev, sevb, k.orow,
                     k.oarea, k.ocode);
  GSJ_LAUNCHED();
  return nsingle + nkeep;
}

// both with the wait between; *single_offs (layers without folding) = the kept candidates' exclusive offsets
uint64_t compact_rows(Context& c, const Layer& PL, const Layer& RL, const uint32_t* pa, const uint32_t* pb, uint64_t np, const RefineParams& rp,
                      const RefineOut& ro, bool no_agg, uint32_t* orow, double* oarea, uint32_t* ocode, const uint64_t** single_offs = nullptr) {
  const Compaction k = compact_enqueue(c, PL, RL, pa, pb, np, rp, ro, no_agg, orow, oarea, ocode);
  k.words.fetch(c);
  GSJ_HIP(hipStreamSynchronize(c.stream));
  if (single_offs) *single_offs = k.offs;
  return compact_finish(c, k);
}

// Sub-batches of at most this many candidates write their rows straight into pinned host memory (at the link's rate: 258k
// rows of 12 bytes in 59 us) instead of copying them once their number is known: one host wait instead of two, and none
// for the refinement where it reads nothing back. Larger ones deliver from device memory, where the copy of all but the
// first rows hides behind the callback's work (deliver_rows). A context without pinned memory copies np rows, an upper
// bound, in the same wait where nothing is folded.
constexpr uint64_t DIRECT_ROWS = 256u << 10;

}  // namespace

void join_run(Context& c, const Layer& PL, const Layer& RL, const gsj_join_opts& o, gsj_rows_cb cb, void* user, gsj_join_stats* st,
              const JoinHooks* hooks) {
  GSJ_REQUIRE(!PL.points && !RL.points, GSJ_E_ARG, "join: both layers must be polygon layers");
  GSJ_REQUIRE(RL.has_bvh, GSJ_E_ARG, "join: build layer has no BVH (call gsj_bvh_build)");
  gsj_join_stats s{};
  if (PL.n == 0 || RL.n == 0) { if (st) *st = s; return; }
  hipStream_t stream = c.stream;
  RefineParams rp;
  rp.want_area = o.want_area ? 1 : 0;
  rp.want_relate = o.want_relate ? 1 : 0;
  rp.snap_half_ulp = o.snap_half_ulp ? 1 : 0;
  const MembersFn none;
  for_each_candidate_batch(c, probes_of(PL), RL.bvh, o.upper != 0, o, s, [&](uint32_t* pa, uint32_t* pb, uint64_t np) {
    if (hooks && hooks->prefilter) {
      WallTimer tp;
      np = hooks->prefilter(pa, pb, np);
      s.compact_ms += tp.ms();
      if (np == 0) return;
    }
    WallTimer t2;
    RefineOut ro;
    ro.isect = c.s_flag.as<uint8_t>(np + 16);
    ro.area = rp.want_area ? c.s_area.as<double>(np + 16) : nullptr;
    ro.ev = rp.want_relate ? c.s_ev.as<double4>(np + 16) : nullptr;
    ro.evb = rp.want_relate ? c.s_evb.as<uint32_t>(np + 16) : nullptr;
    rp.done = hooks && hooks->decide ? hooks->decide(pa, pb, np, ro) : nullptr;
    // no host waits between refinement, compaction and the row copy beyond the ones that read sizes back: the
    // stream orders the work (refine_ms and compact_ms are host times up to those reads; split_wait where there is one)
    const bool folds = !o.no_agg && (PL.poly.pfirst || RL.poly.pfirst);
    const bool direct = !hooks && np <= DIRECT_ROWS && (!c.dev_arena || !folds);
    const bool staged = direct && refine_staged(c, np);   // then nothing is read back before the rows are there
    if (staged) refine_stages(c, PL.poly, RL.poly, pa, pb, np, rp, ro);
    else s.heavy += refine_pairs(c, PL.poly, RL.poly, pa, pb, np, rp, ro, &s);
    const double launch_ms = t2.ms();
    if (!staged) s.refine_ms += launch_ms;
    WallTimer t3;
    if (direct) {
      uint32_t* hrow = c.h_pairs.as<uint32_t>(2 * np);
      double* harea = rp.want_area ? c.h_area.as<double>(np) : nullptr;
      uint32_t* hcode = rp.want_relate ? c.h_code.as<uint32_t>(np) : nullptr;
      const bool pinned = !c.dev_arena;
      uint32_t* orow = pinned ? hrow : c.s_out_a.as<uint32_t>(2 * np + 16);
      double* oarea = !harea ? nullptr : pinned ? harea : c.s_out_area.as<double>(np + 16);
      uint32_t* ocode = !hcode ? nullptr : pinned ? hcode : c.s_out_code.as<uint32_t>(np + 16);
      uint64_t nrows = 0;
      auto rows = [&] {   // compaction and the wait
        const Compaction k = compact_enqueue(c, PL, RL, pa, pb, np, rp, ro, o.no_agg != 0, orow, oarea, ocode);
        k.words.fetch(c);
        if (!pinned) {
          GSJ_HIP(hipMemcpyAsync(hrow, orow, np * 8, hipMemcpyDeviceToHost, stream));
          if (harea) GSJ_HIP(hipMemcpyAsync(harea, oarea, np * 8, hipMemcpyDeviceToHost, stream));
          if (hcode) GSJ_HIP(hipMemcpyAsync(hcode, ocode, np * 4, hipMemcpyDeviceToHost, stream));
        }
        GSJ_HIP(hipStreamSynchronize(stream));
        return k;
      };
      Compaction k = rows();
      uint64_t n_over = 0;
      double span_ms = 0;
      if (staged) {
        WallTimer tf;
        if (refine_stages_finish(c, PL.poly, RL.poly, pa, pb, np, rp, ro, s, n_over, span_ms)) {
          span_ms += tf.ms();
          k = rows();   // the pairs refined since change the rows
        }
      }
      s.heavy += n_over;
      const bool late = k.host_folds();
      nrows = compact_finish(c, k);
      if (late) GSJ_HIP(hipStreamSynchronize(stream));   // the rows folded after the wait
      if (staged) split_wait(s, t2.ms(), launch_ms, span_ms);
      else s.compact_ms += t3.ms();
      s.hits += nrows;
      if (nrows && cb && cb(user, hrow, harea, hcode, (size_t)nrows)) throw Error(GSJ_E_CANCEL, "join cancelled by the row callback");
      return;
    }
    uint32_t* orow = c.s_out_a.as<uint32_t>(2 * np + 16);
    double* oarea = c.s_out_area.as<double>(np + 16);
    uint32_t* ocode = c.s_out_code.as<uint32_t>(np + 16);
    const uint64_t nrows = compact_rows(c, PL, RL, pa, pb, np, rp, ro, o.no_agg != 0, orow, oarea, ocode);
    s.compact_ms += t3.ms();
    s.hits += nrows;
    if (hooks && hooks->on_device && nrows) hooks->on_device(orow, rp.want_area ? oarea : nullptr, nrows);
    if ((hooks && hooks->device_only) || nrows == 0) return;
    uint32_t* hrow = c.h_pairs.as<uint32_t>(2 * nrows);
    double* harea = rp.want_area ? c.h_area.as<double>(nrows) : nullptr;
    uint32_t* hcode = rp.want_relate ? c.h_code.as<uint32_t>(nrows) : nullptr;
    RowPart parts[3] = {{orow, hrow, 8}};
    int np_ = 1;
    if (harea) parts[np_++] = {oarea, harea, 8};
    if (hcode) parts[np_++] = {ocode, hcode, 4};
    const bool stop = deliver_rows(c, parts, np_, nrows, s.copy_ms, [&](uint64_t r, uint64_t n) {
      return cb ? cb(user, hrow + 2 * r, harea ? harea + r : nullptr, hcode ? hcode + r : nullptr, (size_t)n) : 0;
    });
    if (stop) throw Error(GSJ_E_CANCEL, "join cancelled by the row callback");
  }, hooks ? hooks->on_members : none);
  if (st) *st = s;
}

uint64_t compact_single_rows(Context& c, const Layer& PL, const Layer& RL, const uint32_t* pa, const uint32_t* pb, uint64_t np, const RefineParams& rp,
                             const RefineOut& ro, uint32_t* orow, double* oarea, const uint64_t** offs) {
  GSJ_REQUIRE(!PL.poly.pfirst && !RL.poly.pfirst, GSJ_E_INTERNAL, "candidate-ordered rows need layers without parents");
  return compact_rows(c, PL, RL, pa, pb, np, rp, ro, false, orow, oarea, nullptr, offs);
}

bool join_batchable(const Layer& P, const Layer& R, const gsj_join_opts& o) {
  // rows map one to one onto candidates (no piece -> parent folding), so a request's rows are a contiguous run
  return o.has_window && !o.cancel && !P.points && !R.points && R.has_bvh && P.n && R.n && probes_batchable(probes_of(P)) &&
         (o.no_agg || (!P.poly.pfirst && !R.poly.pfirst));
}

bool join_compatible(const gsj_join_opts& a, const gsj_join_opts& b) {
  return a.want_area == b.want_area && a.want_relate == b.want_relate && a.upper == b.upper && a.snap_half_ulp == b.snap_half_ulp &&
         a.no_agg == b.no_agg && a.batch_q == b.batch_q && a.max_pairs == b.max_pairs;
}

void join_batch_run(Context& c, const Layer& PL, const Layer& RL, std::vector<BatchJoin>& reqs) {
  const uint32_t k = (uint32_t)reqs.size();
  GSJ_REQUIRE(k >= 1 && k <= MAX_WINDOWS, GSJ_E_ARG, "batch size out of range");
  const gsj_join_opts& o = *reqs[0].o;
  WindowSet ws;
  ws.k = k;
  for (uint32_t r = 0; r < k; r++) {
    GSJ_REQUIRE(join_batchable(PL, RL, *reqs[r].o) && join_compatible(o, *reqs[r].o), GSJ_E_ARG, "request cannot join this batch");
    for (int j = 0; j < 4; j++) ws.w[r][j] = reqs[r].o->window[j];
  }
  hipStream_t stream = c.stream;
  RefineParams rp;
  rp.want_area = o.want_area ? 1 : 0;
  rp.want_relate = o.want_relate ? 1 : 0;
  rp.snap_half_ulp = o.snap_half_ulp ? 1 : 0;
  gsj_join_stats s{};
  std::vector<uint64_t> cand(k, 0), hits(k, 0);
  for_each_candidate_multi(c, probes_of(PL), RL.bvh, o.upper != 0, o, ws, s, [&](uint32_t* pa, uint32_t* pb, uint64_t np, const SegBounds& sb) {
    for (uint32_t r = 0; r < k; r++) cand[r] += sb.h[r + 1] - sb.h[r];
    WallTimer t2;
    RefineOut ro;
    ro.isect = c.s_flag.as<uint8_t>(np + 16);
    ro.area = rp.want_area ? c.s_area.as<double>(np + 16) : nullptr;
    ro.ev = rp.want_relate ? c.s_ev.as<double4>(np + 16) : nullptr;
    ro.evb = rp.want_relate ? c.s_evb.as<uint32_t>(np + 16) : nullptr;
    s.heavy += refine_pairs(c, PL.poly, RL.poly, pa, pb, np, rp, ro, &s);
    s.refine_ms += t2.ms();
    WallTimer t3;
    uint32_t* orow = c.s_out_a.as<uint32_t>(2 * np + 16);
    double* oarea = c.s_out_area.as<double>(np + 16);
    uint32_t* ocode = c.s_out_code.as<uint32_t>(np + 16);
    const uint64_t* offs = nullptr;
    const uint64_t nrows = compact_rows(c, PL, RL, pa, pb, np, rp, ro, o.no_agg != 0, orow, oarea, ocode, &offs);
    std::vector<uint64_t> rlo(k + 1);
    seg_rows(c, sb, offs, np, nrows, rlo.data());
    s.compact_ms += t3.ms();
    if (nrows == 0) return;
    WallTimer t4;
    uint32_t* hrow = c.h_pairs.as<uint32_t>(2 * nrows);
    double* harea = rp.want_area ? c.h_area.as<double>(nrows) : nullptr;
    uint32_t* hcode = rp.want_relate ? c.h_code.as<uint32_t>(nrows) : nullptr;
    GSJ_HIP(hipMemcpyAsync(hrow, orow, nrows * 8, hipMemcpyDeviceToHost, stream));
    if (harea) GSJ_HIP(hipMemcpyAsync(harea, oarea, nrows * 8, hipMemcpyDeviceToHost, stream));
    if (hcode) GSJ_HIP(hipMemcpyAsync(hcode, ocode, nrows * 4, hipMemcpyDeviceToHost, stream));
    GSJ_HIP(hipStreamSynchronize(stream));
    s.copy_ms += t4.ms();
    for (uint32_t r = 0; r < k; r++) {
      const uint64_t a = rlo[r], n = rlo[r + 1] - rlo[r];
      hits[r] += n;
      BatchJoin& q = reqs[r];
      if (n == 0 || !q.cb || q.rc != GSJ_OK) continue;
      if (q.cb(q.user, hrow + 2 * a, harea ? harea + a : nullptr, hcode ? hcode + a : nullptr, (size_t)n)) q.rc = GSJ_E_CANCEL;
    }
  });
  for (uint32_t r = 0; r < k; r++) {
    if (!reqs[r].st) continue;
    gsj_join_stats& st = *reqs[r].st;
    st = s;
    st.candidates = cand[r];
    st.hits = hits[r];
  }
}

}  // namespace gsj
