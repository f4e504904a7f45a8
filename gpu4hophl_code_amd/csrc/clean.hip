// clean.hip -- canonical repair of a sorted label index on gfx950.
//
// Predicate of the reference's CPU clean, hop_constrained_clean_L
// (CPU_HopHL/include/HBPLL/hop_constrained_two_hop_labels_generation.h:422-511):
// walk L(v) in (hub, hop, dist) order with kept := {}; label (u,h,d) is kept iff
//   min{ d1 + d2 : (w,h1,d1) in L(u), (w,h2,d2) in kept, h1 + h2 <= h } > d.
// The reference runs it with a thread pool, so L(u) may be read before or
// after u itself was cleaned; these kernels read the input L(u), and the
// oracle's tests require both readings to give the same output.
//
// Two passes, exact in every case:
//  1. k_clean_pairs: the predicate with `kept` replaced by every earlier label
//     of v.  That set contains the sequential kept set, so its minima are
//     never larger: when it removes nothing from L(v), the sequential walk
//     keeps every label of v as well.  Pass 1 has no order dependence: it
//     tests the pairs of L(v)'s labels densely against a distance bound and
//     looks L(u) up for the few that pass it; long lists, and few of them, take
//     k_clean_tile.
//  2. k_clean_seq: of vertices where pass 1 would remove something, the labels
//     are decided in rounds that reach exactly what the sequential walk does.
// A K-round, rank-ordered generation already satisfies the predicate (its
// acceptance test is the all-earlier test over the same final lists), so on
// this engine's own output pass 1 removes nothing and pass 2 never runs; the
// clean still verifies every label.
// The reference's GPU clean (Hybrid_Generation_Clean/src/label_clean.cu:73-164)
// uses a dense per-vertex hash of all labels instead; the kept-set form is
// the normative one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "device.hpp"

namespace hsdl {

constexpr uint32_t kSeqThreads = 512;          // pass 2: eight waves per vertex
constexpr uint32_t kSeqBits = 65536;           // labels whose bits its LDS holds
constexpr uint32_t kSeqWords = kSeqBits / 32;
constexpr uint32_t kSeqStage = 4096;           // labels it stages in LDS
constexpr uint32_t kTileThreads = 1024;        // pass 1: sixteen waves per vertex
constexpr uint32_t kTileWindow = 4;            // labels of L(v) per work unit (default)
constexpr uint32_t kMaxWindow = 64;            // largest window
// LDS tile budget: two workgroups per CU share its 160 KB
constexpr uint32_t kTileLdsBytes = 78 * 1024 + 16;
// Indexed LDS tiles (graphs of at most 2^20 vertices): a key slot holds
// hub << kIdxBits | row, and the hub's values for hop budgets 1..K sit in a
// compact row array (one row per distinct hub, not per slot; budget 0 holds
// only v's own hub, which pairs only through a head u > v and which the
// tile leaves out: a list with a hub above its vertex, possible only in
// imported label sets, takes a per-slot tile).
// So the LDS holds 4-byte key slots at load factor <= 1/8 for lists of up to
// about 2,000 hubs, and lists of up to 4,094 hubs at all, instead of 16-byte
// slots at up to 2/3 and lists of up to 2,730 (longer ones went to the
// arena, at 5x the time per label): a wave's probe chain is its longest
// lane's, and chains grow fast with the load factor.  Rows < 2^kIdxBits - 1
// keep a key slot from ever reading as empty (all ones).
constexpr uint32_t kIdxBits = 12;
constexpr uint32_t kIdxRows = (1u << kIdxBits) - 1;
constexpr uint32_t kGroupFast = 4;             // group sizes with the unrolled check

// lower bound of hub w in lab[lo, hi)
__device__ inline uint32_t lb_hub(const unsigned long long *lab, uint32_t lo, uint32_t hi,
                                  uint32_t w) {
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (label_hub(lab[mid]) < w) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// ---------------------------------------------------------------- pass 1
// A label i = (u,h,d) of v falls when an earlier label j = (w,h2,d2) of v has a
// partner (w,h1,d1) in L(u) with h1 <= h - h2 and d1 <= d - d2.  The pairs
// (i, j) of one list are tested densely against a bound that few pass, and
// only those look L(u) up:
//   w < u:  d2 <= d - m(u, h - h2), where m(u, x) is the least distance of
//           L(u)'s labels of hop <= x and hub < u (k_clean_min): whatever the
//           partner is, it is no nearer;
//   w = u:  an earlier label of i's own hub group, at no larger distance.
// Streaming every head's list L(u) through a hash tile of L(v) (k_clean_tile,
// below) reads 174 labels per label of v on R-MAT scale 16 (K = 5); the pairs
// of the same labels are 73 per label before the bound, at three VALU
// instructions per 64 of them, and 7.5 after it.  The bound is that sharp in
// this direction because L(u) is the list of the higher-ranked vertex.
//
// Pairs are walked by hop: the slice's labels are copied in hop order (hub
// order within a hop, k_clean_sort), lanes hold 64 consecutive labels i of it,
// and for each hop x below theirs a wave walks the labels j of hop x, which
// are uniform (scalar loads, 16 or 32 to a load): per j one comparison with
// the lane's packed (hub) limit, one with its distance bound, and a shift into
// a 32-bit mask.  The walk of a hop ends at the largest hub among the lanes.
// The mask's pairs go to a queue in LDS, and every 64 of them search L(u) in
// the index, a pair per lane.
struct Pair32 {
  using T = uint32_t;
  uint32_t hop_bits, dist_bits;
  __device__ T pack(unsigned long long l) const {
    return (label_hub(l) << (hop_bits + dist_bits)) | (label_hop(l) << dist_bits) | label_dist(l);
  }
  __device__ uint32_t hub(T l) const { return l >> (hop_bits + dist_bits); }
  __device__ uint32_t hop(T l) const { return __builtin_amdgcn_ubfe(l, dist_bits, hop_bits); }
  __device__ uint32_t dist(T l) const { return l & ((1u << dist_bits) - 1u); }
  __device__ T below(uint32_t u) const { return u << (hop_bits + dist_bits); }  // labels of hubs < u
};
struct Pair64 {
  using T = unsigned long long;
  __device__ T pack(unsigned long long l) const { return l; }
  __device__ uint32_t hub(T l) const { return label_hub(l); }
  __device__ uint32_t hop(T l) const { return label_hop(l); }
  __device__ uint32_t dist(T l) const { return label_dist(l); }
  __device__ T below(uint32_t u) const { return (unsigned long long)u << 32; }
};

// m[u * K + x - 1], x = 1..K: least distance of L(u)'s labels of hop <= x and
// hub < u (m may be null).  maxima: the longest list and the largest distance, in
// kMaxLines copies 64 bytes apart (an atomic per wave and value on one line took
// 80 us of a 4,096-vertex clean).  A wave per vertex.
constexpr uint32_t kMaxLines = 32, kMaxStride = 16;
__global__ void __launch_bounds__(256) k_clean_min(uint32_t n, uint32_t K,
                                                   const unsigned long long *off,
                                                   const unsigned long long *lab, uint32_t *m,
                                                   uint32_t *maxima) {
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / kWave;
  uint32_t ml = 0, md = 0;
  for (uint32_t u = wave; u < n; u += nwaves) {
    const unsigned long long b = off[u];
    const uint32_t len = (uint32_t)(off[u + 1] - b);
    ml = max(ml, len);
    uint32_t best[kMaxK + 1];
#pragma unroll
    for (uint32_t x = 0; x <= kMaxK; ++x) best[x] = kInf32;
    for (uint32_t j = lane; j < len; j += kWave) {
      const unsigned long long l = lab[b + j];
      const uint32_t h = label_hop(l), d = label_dist(l);
      md = max(md, d);
      if (!m || label_hub(l) >= u) continue;
#pragma unroll
      for (uint32_t x = 0; x <= kMaxK; ++x)
        if (x <= K && x >= h) best[x] = min(best[x], d);
    }
    if (!m) continue;
    uint32_t mine = kInf32;
#pragma unroll
    for (uint32_t x = 1; x <= kMaxK; ++x) {
      if (x > K) continue;
      const uint32_t r = wave_min_u32(best[x]);
      if (lane == x - 1) mine = r;
    }
    if (lane < K) m[(uint64_t)u * K + lane] = mine;
  }
  md = wave_max_u32(md);
  __shared__ uint32_t top[2];
  if (threadIdx.x < 2) top[threadIdx.x] = 0;
  __syncthreads();
  if (lane == 0) {
    atomicMax(&top[0], ml);
    atomicMax(&top[1], md);
  }
  __syncthreads();
  if (threadIdx.x < 2 && top[threadIdx.x])
    atomicMax(&maxima[(blockIdx.x % kMaxLines) * kMaxStride + threadIdx.x], top[threadIdx.x]);
}

// The labels of vertices [v0, v1) in hop order (index order within a hop), from
// out[0], and hcnt[(v - v0) * K + x], x < K: labels of v of hop <= x.  A wave
// per vertex counts its labels' hops, then scatters them.
template <class F>
__global__ void __launch_bounds__(256) k_clean_sort(F f, uint32_t v0, uint32_t v1, uint32_t K,
                                                    const unsigned long long *off,
                                                    const unsigned long long *lab,
                                                    typename F::T *out, uint32_t *hcnt) {
  const uint32_t lane = (uint32_t)lane_id();
  const unsigned long long lt_mask = (1ull << lane) - 1ull;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / kWave;
  const unsigned long long base = off[v0];
  for (uint32_t v = v0 + wave; v < v1; v += nwaves) {
    const unsigned long long b = off[v];
    const uint32_t len = (uint32_t)(off[v + 1] - b);
    uint32_t pos[kMaxK + 1];
#pragma unroll
    for (uint32_t x = 0; x <= kMaxK; ++x) pos[x] = 0;
    for (uint32_t j0 = 0; j0 < len; j0 += kWave) {
      const uint32_t hop = j0 + lane < len ? label_hop(lab[b + j0 + lane]) : kInf32;
#pragma unroll
      for (uint32_t x = 0; x <= kMaxK; ++x)
        if (x <= K) pos[x] += (uint32_t)__popcll(__ballot(hop == x));
    }
    uint32_t run = 0;
#pragma unroll
    for (uint32_t x = 0; x <= kMaxK; ++x) {
      const uint32_t c = pos[x];
      pos[x] = run;
      run += c;
      if (x < K && lane == 0) hcnt[(uint64_t)(v - v0) * K + x] = run;
    }
    for (uint32_t j0 = 0; j0 < len; j0 += kWave) {
      const unsigned long long l = lab[b + min(j0 + lane, len - 1)];
      const uint32_t hop = j0 + lane < len ? label_hop(l) : kInf32;
      uint32_t dst = 0;
#pragma unroll
      for (uint32_t x = 0; x <= kMaxK; ++x) {
        if (x > K) continue;
        const unsigned long long mk = __ballot(hop == x);
        if (hop == x) dst = pos[x] + (uint32_t)__popcll(mk & lt_mask);
        pos[x] += (uint32_t)__popcll(mk);
      }
      if (hop != kInf32) out[b - base + dst] = f.pack(l);
    }
  }
}

// Whether L(u) = lab[lo, lo + len) holds a label of hub w, hop <= x and
// distance <= d (per lane).
__device__ inline bool has_partner(const unsigned long long *__restrict__ lab,
                                   unsigned long long lo, uint32_t len, uint32_t w, uint32_t x,
                                   uint32_t d) {
  const unsigned long long *L = lab + lo;
  uint32_t p = 0, left = len;
  while (left) {
    const uint32_t half = left >> 1;
    if (label_hub(L[p + half]) < w) {
      p += half + 1;
      left -= half + 1;
    } else {
      left = half;
    }
  }
  for (; p < len; ++p) {  // one label per hop, hops ascending
    const unsigned long long l = L[p];
    if (label_hub(l) != w || label_hop(l) > x) return false;
    if (label_dist(l) <= d) return true;
  }
  return false;
}

// The walk of a list is quadratic in its length, and so are its lookups where the
// bound rejects little (a long list whose heads have short ones).  A list goes on
// to the tiles, which take |L(u)| probes per label, once 64 of its labels walk past
// kPairWalk others, or a wave's lookups of 64 pairs pass kPairLooks per 64 labels
// (no list of R-MAT and grid builds of 26 to 311 labels per list does).
// Lists of 16,000 labels over heads of 20, whose pairs all pass the bound and find
// nothing: 64 of them 128 -> 4.7 ms (tiles alone 4.8), 4 of 60,000 1,640 -> 14 (14);
// whose pairs all fail it: 10 -> 4.7 (5.2) and 114 -> 11 (10).
constexpr int32_t kPairWalk = 2048;
constexpr int32_t kPairLooks = 16;
enum : uint32_t { kPairsKeep, kPairsRemove, kPairsLeave };

// Whether some pair of v's labels removes one of the 64 labels from position i0
// of the hop-ordered list L (whole wave).  hc: v's prefix counts; q: the wave's
// queue of 128 entries (position of j << 6 | lane of i); look: lookups the wave has
// left for this list.
template <class F>
__device__ uint32_t chunk_removes(const F &f, uint32_t v, uint32_t K,
                              const unsigned long long *__restrict__ off,
                              const unsigned long long *__restrict__ lab,
                              const typename F::T *__restrict__ L,
                              const uint32_t *__restrict__ hc, const uint32_t *__restrict__ m,
                              uint32_t len, uint32_t i0, lds_ptr<uint32_t> q, int32_t &look,
                              uint64_t &streamed) {
  using T = typename F::T;
  const uint32_t lane = (uint32_t)lane_id();
  const unsigned long long lt_mask = (1ull << lane) - 1ull;
  const T li = L[min(i0 + lane, len - 1)];
  const uint32_t u = f.hub(li), h = f.hop(li), d = f.dist(li);
  const bool act = i0 + lane < len && u != v && h > 0;
  const unsigned long long lo = off[u];
  const uint32_t ulen = (uint32_t)(off[u + 1] - lo);
  const uint32_t hmax = __builtin_amdgcn_readfirstlane(wave_max_u32(act ? h : 0u));
  uint32_t qn = 0;
  bool hit = false;
  int32_t walk = kPairWalk;
  look += (int32_t)kPairLooks;
  auto look_up = [&](uint32_t cnt) {
    --look;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t e = q[lane];
    const int il = (int)(e & 63u);
    const T lj = L[lane < cnt ? e >> 6 : 0u];
    const T pi = __shfl(li, il, kWave);
    const unsigned long long plo = __shfl(lo, il, kWave);
    const uint32_t plen = __shfl(ulen, il, kWave);
    if (lane < cnt && has_partner(lab, plo, plen, f.hub(lj), f.hop(pi) - f.hop(lj),
                                  f.dist(pi) - f.dist(lj)))
      hit = true;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  for (uint32_t x = 0; x < hmax; ++x) {
    const uint32_t zb = x ? hc[x - 1] : 0u, ze = hc[x];
    if (zb == ze) continue;
    const uint32_t mu = act && h > x ? m[(uint64_t)u * K + (h - x - 1)] : kInf32;
    const bool ok = mu <= d;
    if (!__ballot(ok)) continue;
    const uint32_t lim = ok ? d - mu : 0u;
    const T ulim = ok ? f.below(u) : (T)0;  // no label lies below 0
    const T umax = f.below(__builtin_amdgcn_readfirstlane(wave_max_u32(ok ? u : 0u)));
    for (uint32_t j = zb; j < ze; j += 32) {
      const T *Z = L + j;
      if (Z[0] >= umax) break;
      streamed += 32;
      walk -= 32;
      if ((walk | look) < 0) return kPairsLeave;
      uint32_t mask = 0;
#pragma unroll
      for (uint32_t t = 0; t < 32; ++t) {
        const T lj = Z[t];  // past the list's end: padding, masked below
        mask = (mask << 1) | (uint32_t)(lj < ulim && f.dist(lj) <= lim);
      }
      if (ze - j < 32) mask &= ~0u << (32 - (ze - j));
      for (;;) {
        const unsigned long long any = __ballot(mask != 0);
        if (!any) break;
        const uint32_t t = (uint32_t)__builtin_clz(mask | 1u);
        if (mask) {
          q[qn + (uint32_t)__popcll(any & lt_mask)] = (j + t) << 6 | lane;
          mask &= ~(0x80000000u >> t);
        }
        qn += (uint32_t)__popcll(any);
        if (qn >= kWave) {
          look_up(kWave);
          qn -= kWave;
          const uint32_t rest = q[kWave + lane];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          if (lane < qn) q[lane] = rest;
          if (__ballot(hit)) return kPairsRemove;
        }
      }
    }
  }
  if (qn) look_up(qn);
  return __ballot(hit) ? kPairsRemove : kPairsKeep;
}

// Whether two labels of one hub group of v's list [vb, vb + len) remove the
// later one, among the 64 from position i0 (index order; whole wave).
__device__ inline bool group_removes(uint32_t v, const unsigned long long *__restrict__ off,
                                     const unsigned long long *__restrict__ lab,
                                     unsigned long long vb, uint32_t len, uint32_t i0) {
  const uint32_t i = i0 + (uint32_t)lane_id();
  bool hit = false;
  if (i < len) {
    const unsigned long long l = lab[vb + i];
    const uint32_t u = label_hub(l), h = label_hop(l), d = label_dist(l);
    for (uint32_t p = i; u != v && p > 0; --p) {
      const unsigned long long e = lab[vb + p - 1];
      if (label_hub(e) != u) break;
      if (label_dist(e) <= d) {
        const unsigned long long lo = off[u];
        if (has_partner(lab, lo, (uint32_t)(off[u + 1] - lo), u, h - label_hop(e),
                        d - label_dist(e)))
          hit = true;
      }
    }
  }
  return __ballot(hit) != 0;
}

// ctr[0]: redo count, ctr[1]: long lists of the slice, ctr[2]: next vertex of
// the slice (kLong: next entry of `longs`), ctr[4..5]: labels read (u64), ctr[8]:
// lists left to the tiles.
// kLong = false: a wave per vertex, lists of more than kCleanLong labels are
// left in `longs`.  kLong = true: a workgroup per list of `longs`, its waves
// taking the chunks in turn.
// (64 lists of 2,000 labels: a wave each 3.3 ms, a workgroup each 1.0; from 512
// labels on a group build's clean takes 6 % longer.)
constexpr uint32_t kCleanLong = 1024;
constexpr uint32_t kCleanClaim = 4;  // vertices a wave claims at once
template <class F, bool kLong>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8)))
k_clean_pairs(F f, uint32_t v0, uint32_t v1, uint32_t K, const unsigned long long *__restrict__ off,
              const unsigned long long *__restrict__ lab, const typename F::T *__restrict__ srt,
              const uint32_t *__restrict__ hcnt, const uint32_t *__restrict__ m, uint32_t *redo,
              uint32_t *longs, uint32_t *left, uint32_t *ctr) {
  __shared__ uint32_t queue[256 / kWave][2 * kWave];
  __shared__ uint32_t sh_l, sh_c, sh_hit;
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  lds_ptr<uint32_t> q = (lds_ptr<uint32_t>)queue[wib];
  const unsigned long long base = off[v0];
  uint64_t streamed = 0;
  if constexpr (!kLong) {
    for (;;) {
      uint32_t c = 0;
      if (lane == 0) c = atomicAdd(&ctr[2], kCleanClaim);
      c = __builtin_amdgcn_readfirstlane(c);
      if (c >= v1 - v0) break;
      for (uint32_t v = v0 + c; v < min(v1, v0 + c + kCleanClaim); ++v) {
        const unsigned long long vb = off[v];
        const uint32_t len = (uint32_t)(off[v + 1] - vb);
        if (len > kCleanLong) {
          if (lane == 0) longs[atomicAdd(&ctr[1], 1u)] = v;
          continue;
        }
        uint32_t end = kPairsKeep;
        int32_t look = 0;
        for (uint32_t i0 = 0; i0 < len && end == kPairsKeep; i0 += kWave)
          end = group_removes(v, off, lab, vb, len, i0)
                    ? kPairsRemove
                    : chunk_removes(f, v, K, off, lab, srt + (vb - base),
                                    hcnt + (uint64_t)(v - v0) * K, m, len, i0, q, look, streamed);
        if (end == kPairsRemove && lane == 0) redo[atomicAdd(&ctr[0], 1u)] = v;
        if (end == kPairsLeave && lane == 0) left[atomicAdd(&ctr[8], 1u)] = v;
      }
    }
  } else {
    const uint32_t cnt = ctr[1];
    for (;;) {
      if (threadIdx.x == 0) {
        sh_l = atomicAdd(&ctr[2], 1u);
        sh_c = 0;
        sh_hit = 0;
      }
      __syncthreads();
      const uint32_t li = __builtin_amdgcn_readfirstlane(sh_l);
      if (li >= cnt) break;
      const uint32_t v = longs[li];
      const unsigned long long vb = off[v];
      const uint32_t len = (uint32_t)(off[v + 1] - vb);
      int32_t look = 0;
      for (;;) {
        uint32_t c = 0;
        if (lane == 0) c = atomicAdd(&sh_c, 1u);
        c = __builtin_amdgcn_readfirstlane(c);
        const uint32_t seen = __hip_atomic_load(&sh_hit, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_WORKGROUP);
        if ((uint64_t)c * kWave >= len || __builtin_amdgcn_readfirstlane(seen)) break;
        const uint32_t end =
            group_removes(v, off, lab, vb, len, c * kWave)
                ? kPairsRemove
                : chunk_removes(f, v, K, off, lab, srt + (vb - base), hcnt + (uint64_t)(v - v0) * K,
                                m, len, c * kWave, q, look, streamed);
        if (end != kPairsKeep && lane == 0) atomicOr(&sh_hit, end);
      }
      __syncthreads();
      if (threadIdx.x == 0 && sh_hit) {
        if (sh_hit & kPairsRemove)
          redo[atomicAdd(&ctr[0], 1u)] = v;
        else
          left[atomicAdd(&ctr[8], 1u)] = v;
      }
      __syncthreads();
    }
  }
  if (lane == 0 && streamed)
    atomicAdd(reinterpret_cast<unsigned long long *>(ctr) + 2, (unsigned long long)streamed);
}

// ------------------------------------------- pass 1, long lists or few
// Long lists (a mean above kPairMean labels) and few: k_clean_tile, a workgroup of
// sixteen waves per vertex.  It builds a hash tile of L(v) (hub -> per-hop
// prefix minimum distance; in LDS, or in the workgroup's slice of a global arena
// for long lists), then the waves take windows of L(v) in turn, find the windows'
// group heads (hub u), stream the heads' lists L(u), and every element (w,h1,d1)
// with w < u looks w up once in the tile: a group label (u,h,d) falls when d1 +
// tile[w][h - h1] <= d.  Pairs through u itself (earlier labels of the same
// group) are checked directly.  The pair form looks up about a dozen labels per
// label there, at random in lists that no cache holds: R-MAT 262,144 at K = 5
// (672 labels per list) takes 164 ms that way (1.1 TB past L2) against 64 ms with
// tiles, 40,001 vertices (531) 7.4 against 6.3 ms, a group of 65,536 (190) 2.5
// against 3.8 ms, and the 1024 x 1024 grid (66; 8-byte lists) 10.0 against 24.5 ms.
// Few lists keep the tiles as well: a wave per list leaves most of the chip idle
// below some 8,192 lists (1,024 lists of 37 labels 175 us against 110, 4,096 of 69
// 275 against 211 us).
constexpr uint64_t kPairMean = 256;
constexpr uint32_t kPairLists = 8192;
// The heads' lists L(u) are streamed from the index's 8-byte labels, or from
// a 32-bit copy of them (hub | hop | dist fields) when the fields fit one
// word: the first pass reads far more list labels than anything else and
// runs near the rate HBM sustains, so half the bytes is what counts.
struct Stream64 {
  using T = unsigned long long;
  const unsigned long long *lab;
  __device__ const T *list(unsigned long long b) const { return lab + b; }
  // elements of L(u) of hop <= maxhop: the whole list (not hop-sorted)
  __device__ uint32_t upto(uint32_t, uint32_t, uint32_t len) const { return len; }
  __device__ void dec(T l, uint32_t &w, uint32_t &h, uint32_t &d) const {
    w = label_hub(l);
    h = label_hop(l);
    d = label_dist(l);
  }
};
// The 32-bit copy keeps each list stably sorted by hop (hub order within a
// hop), with hcnt[u * K + x] = elements of L(u) of hop <= x (x < K): an element pairs with the tile through hop h1 + 1 or more
// when w != v, so a group whose deepest label has hop maxh can use only
// L(u)'s elements of hop <= maxh - 1 -- a prefix of the sorted list, which
// the stream stops at (the self label, hop 0, is its first element).  Only a
// head u above v can hold w = v (pairing with v's self label, hop 0): its
// stream goes to hop maxh.
struct Stream32 {
  using T = uint32_t;
  const uint32_t *lab;
  uint32_t hop_bits, dist_bits;
  const uint32_t *hcnt;
  uint32_t K;
  __device__ const T *list(unsigned long long b) const { return lab + b; }
  __device__ uint32_t upto(uint32_t u, uint32_t maxhop, uint32_t len) const {
    return maxhop < K ? hcnt[(uint64_t)u * K + maxhop] : len;
  }
  __device__ void dec(T l, uint32_t &w, uint32_t &h, uint32_t &d) const {
    w = l >> (hop_bits + dist_bits);
    h = __builtin_amdgcn_ubfe(l, dist_bits, hop_bits);
    d = l & ((1u << dist_bits) - 1u);
  }
};

// True when the all-earlier predicate removes a label of a group whose head
// lies in L(v)[p0, p0 + win).  The wave walks the window's heads in order
// (uniform control flow: the group's labels are uniform scalar loads) and
// streams each head's list L(u) 128 elements per step with coalesced loads;
// only the filter and the tile probe are per lane.  The two step buffers
// alternate (a, b) and loads are clamped to the list (lanes past the end are
// masked), so a step's probes run while the next step's loads are in flight.
// KP / VP: the tile's address space (LDS or the global arena).
template <class V, bool kIdx, class S, class KP, class VP>
__device__ bool window_removes(uint32_t v, uint32_t K1, const unsigned long long *__restrict__ off,
                               const S &str, const unsigned long long *__restrict__ Lv, uint32_t len,
                               uint32_t p0, uint32_t win, KP keys, VP vals, uint32_t cap,
                               uint32_t last_row, uint64_t &streamed) {
  constexpr bool kArena = !std::is_same<KP, lds_ptr<uint32_t>>::value;
  // hub w's key slot: sets `found` and returns the index of its value row
  // (an empty slot's is any in-bounds row: the caller masks it)
  auto find = [&](uint32_t w, bool &found) -> uint32_t {
    uint32_t slot = hash_slot(w, cap);
    uint32_t k = keys[slot];
    if (kIdx) {
      while ((k >> kIdxBits) != w && k != kInf32) {
        slot = (slot + 1) & (cap - 1);
        k = keys[slot];
      }
      // an empty slot reads hub 2^20 - 1, which ranks below every head u
      // that the pair test also asks for (w < u)
      found = (k >> kIdxBits) == w;
      return mul_u24(min(k & kIdxRows, last_row), K1 - 1);
    }
    while (k != w && k != kInf32) {
      slot = (slot + 1) & (cap - 1);
      k = keys[slot];
    }
    found = k == w;
    return mul_u24(slot, K1);
  };
  // the value of row `base` for a group label of hop g and an element of hop
  // h1 (budget x = g - h1), and whether the budget can pair (reach): per-slot
  // rows hold budgets 0..K, indexed rows 1..K (budget 0 holds only v's hub)
  auto value_at = [&](uint32_t base, uint32_t g, uint32_t h1, bool &reach) -> uint32_t {
    if (kIdx) {
      reach = g > h1;
      return vals[base + (reach ? g - 1u - h1 : 0u)];
    }
    reach = g >= h1;
    return vals[base + (reach ? g - h1 : 0u)];
  };
  const uint32_t lane = (uint32_t)lane_id();
  bool hit = false;
  const uint32_t pend = min(p0 + win, len);
  for (uint32_t p = p0; p < pend; ++p) {
    const uint32_t u = label_hub(Lv[p]);
    if ((p > 0 && label_hub(Lv[p - 1]) == u) || u == v) continue;  // not a head / self label
    uint32_t glen = 0, maxh = 0, maxd = 0;
    while (p + glen < len && label_hub(Lv[p + glen]) == u) {
      const unsigned long long g = Lv[p + glen];
      maxh = max(maxh, label_hop(g));
      maxd = max(maxd, label_dist(g));
      ++glen;
    }
    const unsigned long long ub = off[u];
    // an element (w,h1,d1) of L(u) pairs with the tile through hop >= h1 + 1
    // when w != v; w = v (possible only for u > v, in imported label sets
    // whose hubs may rank below their vertex) pairs with v's self label
    const uint32_t hmin = u > v ? 0u : 1u;
    const uint32_t ulen = str.upto(u, maxh - hmin, (uint32_t)(off[u + 1] - ub));
    if (ulen == 0) continue;
    const typename S::T *Lu = str.list(ub);
    // the group's hops and distances, decoded once per head into scalars for
    // groups of up to kGroupFast labels (a group holds at most K + 1, one per
    // hop): the per-element loop over them is then unrolled straight-line
    // code instead of a scalar load, a wait and a decode per group label
    const bool fast = glen <= kGroupFast;
    uint32_t gh[kGroupFast], gd[kGroupFast];
#pragma unroll
    for (uint32_t t = 0; t < kGroupFast; ++t) {
      const unsigned long long g = (fast && t < glen) ? Lv[p + t] : 0ull;
      gh[t] = label_hop(g);
      gd[t] = label_dist(g);
    }
    streamed += ulen;
    const uint32_t last = ulen - 1;
    // one element (w,h1,d1) of L(u) against the group.  The pass issues
    // VALU instructions near the rate a CU sustains, so the check is
    // straight-line code but for the rare collision chain:
    // * a lane past the list's end holds a copy of its last element, which
    //   gives the same answer as the element itself: no mask;
    // * in an LDS tile the lookup runs for every lane: the chain ends at w
    //   or at an empty slot (whose values count only when k == w), and the
    //   shortcuts d1 <= maxd and h1 + hmin <= maxh are left to the pair test,
    //   which implies them (d1 + m <= gd with m >= 0; budget gh - h1 = 0
    //   holds only v's self label, hop-0 labels being self labels); an arena
    //   tile's lookups are global loads, which the shortcuts still save;
    // * a 16-bit empty value (0xFFFF) is above every label distance (small
    //   values: the largest distance < 0xFFFF), so only 32-bit values test
    //   for it.
    auto check = [&](typename S::T l) {
      uint32_t w, h1, d1;
      str.dec(l, w, h1, d1);
      if (w == u) {
        // through hub u: earlier labels of the group against later ones
        for (uint32_t t1 = 0; t1 < glen; ++t1) {
          const unsigned long long g1 = Lv[p + t1];
          for (uint32_t t2 = t1 + 1; t2 < glen; ++t2) {
            const unsigned long long g2 = Lv[p + t2];
            if (h1 + label_hop(g1) <= label_hop(g2) && d1 + label_dist(g1) <= label_dist(g2))
              hit = true;
          }
        }
      }
      if (kArena && !((w < u) & (h1 + hmin <= maxh) & (d1 <= maxd))) return;
      bool found;
      const uint32_t base = find(w, found);
      const bool pair = found & (w < u);
      auto fits = [&](uint32_t m, uint32_t gd) -> bool {
        if (sizeof(V) == 2) return d1 + m <= gd;
        return (m != TileVal<V>::kEmpty) & (d1 + m <= gd);
      };
      if (fast) {
#pragma unroll
        for (uint32_t t = 0; t < kGroupFast; ++t) {
          if (t >= glen) break;
          // a label shallower than h1 reads the row's first value and is
          // masked; at equal hops only the hop-0 tile label (v's) pairs
          bool reach;
          const uint32_t m = value_at(base, gh[t], h1, reach);
          hit |= pair & reach & fits(m, gd[t]);
        }
      } else {
        for (uint32_t t = 0; t < glen; ++t) {
          const unsigned long long g = Lv[p + t];
          const uint32_t hg = label_hop(g);
          bool reach;
          const uint32_t m = value_at(base, hg, h1, reach);
          if (pair && reach && fits(m, label_dist(g))) hit = true;
        }
      }
    };
    // a group of one label (most groups): its hop and distance are the
    // group's maxima, no pair runs through u inside the group, and the
    // per-label loop and its branches go
    auto check1 = [&](typename S::T l) {
      uint32_t w, h1, d1;
      str.dec(l, w, h1, d1);
      if (kArena && !((w < u) & (h1 + hmin <= maxh) & (d1 <= maxd))) return;
      bool found, reach;
      const uint32_t base = find(w, found);
      const uint32_t m = value_at(base, gh[0], h1, reach);
      const bool near = sizeof(V) == 2 ? d1 + m <= gd[0]
                                       : (m != TileVal<V>::kEmpty) & (d1 + m <= gd[0]);
      hit |= found & (w < u) & reach & near;
    };
    auto ld = [&](uint32_t j) { return Lu[min(j, last)]; };
    auto stream = [&](auto &&chk) {
      typename S::T a0 = ld(lane), a1 = ld(kWave + lane);
      for (uint32_t jb = 0; jb < ulen; jb += 4 * kWave) {
        const typename S::T b0 = ld(jb + 2 * kWave + lane), b1 = ld(jb + 3 * kWave + lane);
        chk(a0);
        chk(a1);
        if (jb + 2 * kWave >= ulen) break;
        a0 = ld(jb + 4 * kWave + lane);
        a1 = ld(jb + 5 * kWave + lane);
        chk(b0);
        chk(b1);
      }
    };
    if (glen == 1)
      stream(check1);
    else
      stream(check);
  }
  return __ballot(hit) != 0;
}

// Builds the tile of L(v) (keys, vals in LDS or in the workgroup's arena
// slice) and runs the windows of L(v) over it; true when some window removes
// a label.  Whole workgroup.
template <class V, bool kIdx, class S, class KP, class VP>
__device__ __attribute__((always_inline)) inline bool clean_vertex(
    uint32_t v, uint32_t K1, const unsigned long long *__restrict__ off, const S &str,
    const unsigned long long *__restrict__ Lv,
    uint32_t len, KP keys, VP vals, uint32_t cap, uint32_t rows, bool in_arena, uint32_t win,
    uint32_t &sh_win, uint32_t &sh_removed, uint32_t &sh_row, uint64_t &streamed) {
  const uint32_t tid = threadIdx.x, lane = (uint32_t)lane_id();
  for (uint32_t i = tid; i < cap; i += kTileThreads) keys[i] = kInf32;
  if (tid == 0) sh_row = 0;
  __syncthreads();
  // one thread per group: claim the hub's slot (and, indexed, a value row),
  // write its per-hop prefix minima
  for (uint32_t i = tid; i < len; i += kTileThreads) {
    const uint32_t w = label_hub(Lv[i]);
    if (i > 0 && label_hub(Lv[i - 1]) == w) continue;
    if (kIdx && w == v) continue;  // v's own hub: no head u > v pairs with it here
    uint32_t slot = hash_slot(w, cap);
    if (kIdx) {
      const uint32_t row = atomicAdd(&sh_row, 1u);
      while (atomicCAS((uint32_t *)&keys[slot], kInf32, (w << kIdxBits) | row) != kInf32)
        slot = (slot + 1) & (cap - 1);
      slot = row;  // the values go to the row
    } else {
      while (atomicCAS((uint32_t *)&keys[slot], kInf32, w) != kInf32) slot = (slot + 1) & (cap - 1);
    }
    uint32_t m[kMaxK + 1];
#pragma unroll
    for (uint32_t x = 0; x <= kMaxK; ++x) m[x] = kInf32;
    for (uint32_t q = i; q < len && label_hub(Lv[q]) == w; ++q) {
      const uint32_t h = label_hop(Lv[q]), d = label_dist(Lv[q]);
#pragma unroll
      for (uint32_t x = 0; x <= kMaxK; ++x)
        if (x == h) m[x] = min(m[x], d);
    }
    uint32_t run = kInf32;
#pragma unroll
    for (uint32_t x = 0; x <= kMaxK; ++x) {
      run = min(run, m[x]);
      const V val = (V)min(run, (uint32_t)TileVal<V>::kEmpty);
      if (kIdx) {
        if (x >= 1 && x < K1) vals[slot * (K1 - 1) + (x - 1)] = val;  // budgets 1..K
      } else {
        if (x < K1) vals[slot * K1 + x] = val;
      }
    }
  }
  // an arena tile was written through L2: drop stale L1 lines before reading
  if (in_arena) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __syncthreads();
  if (in_arena) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  for (;;) {
    uint32_t p0 = 0;
    if (lane == 0) p0 = atomicAdd(&sh_win, win);
    p0 = __builtin_amdgcn_readfirstlane(__shfl(p0, 0, kWave));
    if (p0 >= len) break;
    if (window_removes<V, kIdx>(v, K1, off, str, Lv, len, p0, win, keys, vals, cap, rows - 1,
                                streamed)) {
      if (lane == 0) sh_removed = 1;
      break;
    }
  }
  __syncthreads();
  return sh_removed != 0;
}

// The n vertices from 0, or those of `list`.  ctr[0]: redo count, ctr[2]: next vertex, ctr[4..5]: labels of L(u) read (u64).  gtile: per-workgroup arena slices
// of gwords words for tiles above lds_slots slots.
template <class V, class S>
__global__ void __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(8)))
k_clean_tile(uint32_t n, const uint32_t *list, uint32_t K, const unsigned long long *__restrict__ off,
             const unsigned long long *__restrict__ lab, S str,
             uint32_t *redo, uint32_t *ctr, uint32_t lds_slots, uint32_t *gtile,
             uint64_t gwords, uint32_t win, uint32_t indexed) {
  extern __shared__ uint32_t lds[];
  __shared__ uint32_t sh_v, sh_win, sh_heads, sh_removed, sh_row;
  // LDS bytes for a tile (the launch gives lds_slots slots of key + values)
  const uint32_t lds_tile_bytes = lds_slots * (4u + (K + 1) * (uint32_t)sizeof(V));
  const uint32_t K1 = K + 1;
  const uint32_t tid = threadIdx.x, lane = (uint32_t)lane_id();
  uint32_t *gkeys = gtile + (uint64_t)blockIdx.x * gwords;
  uint64_t streamed = 0;  // labels of L(u) lists this wave read
  for (;;) {
    if (tid == 0) {
      sh_v = atomicAdd(&ctr[2], 1u);
      sh_win = 0;
      sh_heads = 0;
      sh_removed = 0;
    }
    __syncthreads();
    // wave-uniform values are made explicit, so the list offsets and hubs are
    // scalar loads and the loops over them carry no per-lane masks
    const uint32_t next = __builtin_amdgcn_readfirstlane(sh_v);
    if (next >= n) break;
    const uint32_t v = list ? list[next] : next;
    const unsigned long long vb = off[v];
    const uint32_t len = (uint32_t)(off[v + 1] - vb);
    const unsigned long long *Lv = lab + vb;
    if (len > 1) {
      // distinct hubs of L(v) size the tile
      uint32_t mine = 0;
      for (uint32_t i = tid; i < len; i += kTileThreads)
        mine += (i == 0 || label_hub(Lv[i]) != label_hub(Lv[i - 1])) ? 1u : 0u;
      mine = wave_sum_u32(mine);
      if (lane == 0 && mine) atomicAdd(&sh_heads, mine);
      __syncthreads();
      const uint32_t heads = sh_heads;
      const uint32_t cap = tile_cap_for(heads);
      // indexed: key slots at load factor <= 1/8 where the rows leave room
      uint32_t icap = 0;
      // (lists are hub-sorted: the last hub is the largest)
      if (indexed && heads <= kIdxRows && label_hub(Lv[len - 1]) <= v) {
        const uint32_t row_bytes = (heads * K * (uint32_t)sizeof(V) + 15u) & ~15u;
        if (row_bytes + 4u * cap <= lds_tile_bytes) {
          icap = pow2_at_least(8ull * heads + 4);
          while (row_bytes + 4u * icap > lds_tile_bytes) icap >>= 1;
        }
      }
      if (icap) {
        clean_vertex<V, true>(v, K1, off, str, Lv, len, (lds_ptr<uint32_t>)lds,
                              (lds_ptr<V>)(lds + icap), icap, heads, false, win, sh_win,
                              sh_removed, sh_row, streamed);
      } else if (cap <= lds_slots) {
        const uint32_t lcap = lds_tile_cap(heads, lds_slots);
        clean_vertex<V, false>(v, K1, off, str, Lv, len, (lds_ptr<uint32_t>)lds,
                               (lds_ptr<V>)(lds + lcap), lcap, lcap, false, win, sh_win,
                               sh_removed, sh_row, streamed);
      } else {
        clean_vertex<V, false>(v, K1, off, str, Lv, len, (glb_ptr<uint32_t>)gkeys,
                               (glb_ptr<V>)(gkeys + cap), cap, cap, true, win, sh_win,
                               sh_removed, sh_row, streamed);
      }
    }
    if (sh_removed && tid == 0) redo[atomicAdd(&ctr[0], 1u)] = v;
    __syncthreads();  // shared state and the tile are reused for the next vertex
  }
  if (lane == 0 && streamed)
    atomicAdd(reinterpret_cast<unsigned long long *>(ctr) + 2, (unsigned long long)streamed);
}

// Pass 2's start: every label kept, every length the old one.
__global__ void k_clean_keep_all(uint32_t n, const unsigned long long *off, uint32_t *new_len) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x)
    new_len[v] = (uint32_t)(off[v + 1] - off[v]);
}

// ---------------------------------------------------------------- pass 2
// The reference's sequential walk for the vertices in `list`, decided in rounds
// instead of in order.  A label is kept when no pair with earlier labels that may
// still be kept removes it, and falls when a pair with one that is known to be
// kept does; either is what the walk decides, whose kept set lies between the
// two.  The first label left open by a round has only decided ones before it, so
// a round decides at least that one; nearly all are decided by the first two.
// A workgroup of eight waves per vertex: the waves take windows of L(v) in
// turn, and for a group of hub u (with an open label) the 64 lanes stream L(u);
// each lane searches its label's hub w < u in L(v) and folds the pairs into
// per-hop minima m[x] (x = h1 + h2), one set over the labels that may be kept and
// one over those that are.  A wave min-reduction and a prefix-min over x give the
// best pair for every hop budget; the group's labels are then decided in hop
// order, adding the pairs through hub u itself.
// What binds is the searches' latency: eight waves with a list in 48 KB of LDS, three
// workgroups per CU.  Walking a list in order, a wave per list, took its groups'
// chains of round trips one after the other: 3,001 vertices with redundant labels
// 2.03 ms, most of it the longest lists', against 0.74 ms (sixteen waves, one
// workgroup per CU: 1.14; lists dealt out instead of claimed: 0.90).
// kLong = false: lists of up to kSeqBits labels, their kept and fallen bits in
// LDS (and the list itself up to kSeqStage labels); longer lists are left to the
// kLong = true launch, whose bits live in the workgroup's slice of `gbits` (2 *
// gwords words): read and written with agent-scope atomics, so every wave sees the
// others' updates without relying on the vector L1.  A hub group of more than 32
// labels (impossible with one label per (hub, hop) and K <= 15, which import and
// generation guarantee) sets bad bit 2 instead of overflowing the group's mask.
template <bool kLong>
__global__ void __launch_bounds__(kSeqThreads) k_clean_seq(
    uint32_t K, const unsigned long long *off, const unsigned long long *lab, uint8_t *keep,
    uint32_t *new_len, const uint32_t *list, const uint32_t *list_cnt, uint32_t *next_list,
    uint32_t *bad, uint32_t *gbits, uint32_t gwords) {
  __shared__ unsigned long long stage[kLong ? 1 : kSeqStage];
  __shared__ uint32_t bits[kLong ? 1 : 2 * kSeqWords];  // kept, then fallen
  // a round's next window and whether it leaves labels open: three sets in turn,
  // the next round's cleared while this one runs, so that nothing is reset where
  // the rounds' loop turns
  __shared__ uint32_t sh_next[3], sh_open[3];
  __shared__ uint32_t sh_bad, sh_kept, sh_list;
  const uint32_t tid = threadIdx.x, lane = (uint32_t)lane_id();
  const uint32_t words_max = kLong ? gwords : kSeqWords;
  uint32_t *const slice = kLong ? gbits + (uint64_t)blockIdx.x * 2 * gwords : bits;
  // 32 bits of a set from position i on (fallen: set 1)
  auto word = [&](uint32_t set, uint32_t i) -> uint32_t {
    uint32_t *w = slice + set * words_max + i;
    if constexpr (kLong)
      return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto bit = [&](uint32_t set, uint32_t i) { return (word(set, i >> 5) >> (i & 31)) & 1u; };
  auto put = [&](uint32_t set, uint32_t i) {
    atomicOr(slice + set * words_max + (i >> 5), 1u << (i & 31));
  };
  // every value that decides a loop with barriers in it is made scalar: the
  // compiler then branches for the whole wave, never for some of its lanes
  const uint32_t cnt = __builtin_amdgcn_readfirstlane(*list_cnt);
  // a workgroup's first list is its own id, later ones come from a counter
  auto claim = [&]() {
    __syncthreads();  // the shared state is the next list's
    if (tid == 0) sh_list = gridDim.x + atomicAdd(next_list, 1u);
    __syncthreads();
    return (uint32_t)__builtin_amdgcn_readfirstlane(sh_list);
  };
  for (uint32_t li = blockIdx.x; li < cnt; li = claim()) {
    const uint32_t v = __builtin_amdgcn_readfirstlane(list[li]);
    const unsigned long long vb = off[v];
    const uint32_t len = __builtin_amdgcn_readfirstlane((uint32_t)(off[v + 1] - vb));
    const unsigned long long *Lv = lab + vb;
    if (kLong ? (len <= kSeqBits) : (len > kSeqBits)) continue;  // the other launch's
    const uint32_t words = (len + 31) / 32;
    if (kLong && words > gwords) {
      if (tid == 0) atomicOr(bad, 1u);
      continue;
    }
    for (uint32_t i = tid; i < 2 * words; i += kSeqThreads) {
      uint32_t *w = slice + (i < words ? i : words_max + i - words);
      if constexpr (kLong)
        __hip_atomic_store(w, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        *w = 0;
    }
    const bool staged = !kLong && len <= kSeqStage;
    if (staged)
      for (uint32_t i = tid; i < len; i += kSeqThreads) stage[i] = Lv[i];
    const lds_ptr<const unsigned long long> Sv = (lds_ptr<const unsigned long long>)stage;
    auto at = [&](uint32_t i) -> unsigned long long {
      if (staged) return Sv[i];
      return Lv[i];
    };
    if (tid < 3) sh_next[tid] = sh_open[tid] = 0;
    if (tid == 0) sh_bad = sh_kept = 0;
    __syncthreads();
    for (uint32_t round = 0;; round = round == 2 ? 0 : round + 1) {
      // (last read before the barrier that ended the round before this one)
      if (tid == 0) sh_next[round == 2 ? 0 : round + 1] = sh_open[round == 2 ? 0 : round + 1] = 0;
      for (;;) {
        uint32_t p0 = 0;
        if (lane == 0) p0 = atomicAdd(&sh_next[round], kTileWindow);
        p0 = __builtin_amdgcn_readfirstlane(p0);
        if (p0 >= len) break;
        for (uint32_t gb = p0; gb < min(len, p0 + kTileWindow); ++gb) {
          const uint32_t u = __builtin_amdgcn_readfirstlane(label_hub(at(gb)));
          if (gb > 0 && label_hub(at(gb - 1)) == u) continue;  // not a group's head
          // the group [gb, ge) of at most K + 1 labels, the most its labels allow,
          // and what is decided of it
          uint32_t ge = gb, maxd = 0, maxh = 0, kept = 0, fell = 0;
          while (ge < len && ge - gb <= 32 && label_hub(at(ge)) == u) {
            if (ge - gb < 32) {
              kept |= bit(0, ge) << (ge - gb);
              fell |= bit(1, ge) << (ge - gb);
            }
            maxd = max(maxd, label_dist(at(ge)));
            maxh = max(maxh, label_hop(at(ge)));
            ++ge;
          }
          const uint32_t size = ge - gb;
          if (size > 32) {  // see above: cannot happen on valid input
            if (lane == 0) atomicOr(&sh_bad, 2u);
            continue;
          }
          const uint32_t all = size == 32 ? ~0u : (1u << size) - 1u;
          if ((kept | fell) == all) continue;
          uint32_t ma[kMaxK + 1], mk[kMaxK + 1];
#pragma unroll
          for (uint32_t x = 0; x <= kMaxK; ++x) ma[x] = mk[x] = kInf32;
          const unsigned long long ub = off[u];
          const uint32_t ulen = (uint32_t)(off[u + 1] - ub);
          const unsigned long long *Lu = lab + ub;
          for (uint32_t j = lane; gb > 0 && j < ulen; j += kWave) {
            const unsigned long long l = Lu[j];
            const uint32_t w = label_hub(l), h1 = label_hop(l), d1 = label_dist(l);
            if (w >= u || h1 > maxh || d1 > maxd) continue;
            uint32_t p = 0, hi = gb;
            while (p < hi) {
              const uint32_t mid = (p + hi) >> 1;
              if (label_hub(at(mid)) < w) p = mid + 1; else hi = mid;
            }
            for (; p < gb; ++p) {
              const unsigned long long q = at(p);
              if (label_hub(q) != w) break;
              const uint32_t x = h1 + label_hop(q), sum = d1 + label_dist(q);
              if (x > maxh || sum > maxd || bit(1, p)) continue;
              const bool sure = bit(0, p);
#pragma unroll
              for (uint32_t y = 0; y <= kMaxK; ++y)
                if (y == x) {
                  ma[y] = min(ma[y], sum);
                  if (sure) mk[y] = min(mk[y], sum);
                }
            }
          }
          // L(u)'s own labels (hub u): found by search, since a list may also
          // hold hubs ranked below its vertex (imported label sets)
          const uint32_t ub0 = lb_hub(Lu, 0, ulen, u);
          uint32_t ra = kInf32, rk = kInf32;
#pragma unroll
          for (uint32_t x = 0; x <= kMaxK; ++x) {
            if (x <= K) {
              ra = min(ra, wave_min_u32(ma[x]));
              rk = min(rk, wave_min_u32(mk[x]));
            }
            ma[x] = ra;
            mk[x] = rk;
          }
          // decide the group's open labels in order (all lanes compute the same)
          uint32_t nk = 0, nf = 0;
          for (uint32_t i = 0; i < size; ++i) {
            if (((kept | fell) >> i) & 1u) continue;
            const unsigned long long l = at(gb + i);
            const uint32_t h = label_hop(l), d = label_dist(l);
            uint32_t best_any = kInf32, best_kept = kInf32;
#pragma unroll
            for (uint32_t x = 0; x <= kMaxK; ++x)
              if (x == h) {
                best_any = ma[x];
                best_kept = mk[x];
              }
            // pairs through hub u: L(u)'s hub-u labels x earlier labels of this group
            for (uint32_t k2 = 0; k2 < i; ++k2) {
              if (((fell | nf) >> k2) & 1u) continue;
              const bool sure = ((kept | nk) >> k2) & 1u;
              const unsigned long long q = at(gb + k2);
              for (uint32_t t = ub0; t < ulen; ++t) {
                const unsigned long long r = Lu[t];
                if (label_hub(r) != u) break;
                if (label_hop(r) + label_hop(q) > h) continue;
                const uint32_t sum = label_dist(r) + label_dist(q);
                best_any = min(best_any, sum);
                if (sure) best_kept = min(best_kept, sum);
              }
            }
            if (best_any > d)
              nk |= 1u << i;
            else if (best_kept <= d)
              nf |= 1u << i;
          }
          if (lane < size && ((nk >> lane) & 1u)) put(0, gb + lane);
          if (lane < size && ((nf >> lane) & 1u)) put(1, gb + lane);
          if (lane == 0 && (kept | fell | nk | nf) != all) atomicOr(&sh_open[round], 1u);
        }
      }
      __syncthreads();
      // (a group too large is met in the first round: no later one sets sh_bad)
      if (!__builtin_amdgcn_readfirstlane(sh_open[round] && !sh_bad)) break;
    }
    if (__builtin_amdgcn_readfirstlane(sh_bad)) {
      if (tid == 0) atomicOr(bad, sh_bad);
    } else {
      uint32_t k = 0;
      for (uint32_t i = tid; i < len; i += kSeqThreads) {
        const uint32_t one = bit(0, i);
        keep[vb + i] = (uint8_t)one;
        k += one;
      }
      k = wave_sum_u32(k);
      if (lane == 0 && k) atomicAdd(&sh_kept, k);
      __syncthreads();
      if (tid == 0) new_len[v] = sh_kept;
    }
  }
}

// Kept labels (and their parents, when par is not null) into the new CSR.
__global__ void __launch_bounds__(256) k_compact(uint32_t n, const unsigned long long *off,
                                                 const unsigned long long *lab,
                                                 const uint8_t *keep,
                                                 const unsigned long long *noff,
                                                 unsigned long long *nlab,
                                                 const uint32_t *par, uint32_t *npar) {
  const int lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / kWave;
  const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (uint32_t v = wave; v < n; v += nwaves) {
    const unsigned long long b = off[v], e = off[v + 1];
    unsigned long long dst = noff[v];
    for (unsigned long long i = b; i < e; i += kWave) {
      const bool valid = i + lane < e;
      const bool k = valid && keep[i + lane];
      const unsigned long long mk = __ballot(k);
      if (k) {
        nlab[dst + __popcll(mk & lt)] = lab[i + lane];
        if (par) npar[dst + __popcll(mk & lt)] = par[i + lane];
      }
      dst += __popcll(mk);
    }
  }
}

// The clean's working buffers (the hop-ordered copy and its counts, the least
// distances, keep flags, lengths) and the index arrays a clean replaces are kept
// per device for the next clean, sized for the largest so far: freeing and
// allocating gigabytes inside every clean now and then cost a tenth of a
// second there.  hsdl_release_scratch frees them.
enum CleanScratchId : int {
  kCsKeep, kCsNewLen, kCsRedo, kCsSrt, kCsHcnt, kCsMins, kCsLongs, kCsCtr, kCsGtile, kCsOff,
  kCsLab, kCsCount
};
constexpr int kCsDevices = 64;
struct CleanScratch {
  void *p[kCsCount] = {};
  size_t bytes[kCsCount] = {};
};
static CleanScratch g_clean_scratch[kCsDevices];
static std::mutex g_clean_scratch_mu;

// b <- a kept buffer of at least n bytes when there is one, else a new one
static int take_scratch(int dev, int id, DevBuf &b, size_t n) {
  if (dev >= 0 && dev < kCsDevices) {
    std::lock_guard<std::mutex> lk(g_clean_scratch_mu);
    CleanScratch &c = g_clean_scratch[dev];
    if (c.p[id] && c.bytes[id] >= n) {
      b.release();
      b.p = c.p[id];
      b.bytes = c.bytes[id];
      c.p[id] = nullptr;
      c.bytes[id] = 0;
      return HSDL_OK;
    }
    if (c.p[id]) {
      (void)hipFree(c.p[id]);
      c.p[id] = nullptr;
      c.bytes[id] = 0;
    }
  }
  return b.alloc(n);
}
// b goes back to the device's kept buffers (or is freed when the slot is taken)
static void give_scratch(int dev, int id, DevBuf &b) {
  if (!b.p || dev < 0 || dev >= kCsDevices) return;
  std::lock_guard<std::mutex> lk(g_clean_scratch_mu);
  CleanScratch &c = g_clean_scratch[dev];
  if (c.p[id]) return;  // b frees itself
  c.p[id] = b.p;
  c.bytes[id] = b.bytes;
  b.p = nullptr;
  b.bytes = 0;
}

int clean_index(hsdl_index *idx) {
  int rc = use_device(idx->device, nullptr);
  if (rc) return rc;
  const uint32_t n = idx->n;
  const uint64_t t0 = now_ns();
  hipStream_t st;
  HSDL_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  struct G {
    hipStream_t s;
    ~G() { (void)hipStreamDestroy(s); }
  } guard{st};
  DevBuf keep, new_len, noff, nlab, redo, ctr, srt, hcnt, mins, longs, gtile;
  const int dev = idx->device;
  // every buffer taken from the kept ones goes back when the clean ends (a clean
  // that failed may have kernels in flight on them)
  struct Give {
    hipStream_t st;
    int dev;
    DevBuf *b[9];
    int id[9];
    bool idle = false;
    ~Give() {
      if (!idle) (void)hipStreamSynchronize(st);
      for (int i = 0; i < 9; ++i) give_scratch(dev, id[i], *b[i]);
    }
  } give{st, dev, {&keep, &new_len, &redo, &srt, &hcnt, &mins, &longs, &ctr, &gtile},
         {kCsKeep, kCsNewLen, kCsRedo, kCsSrt, kCsHcnt, kCsMins, kCsLongs, kCsCtr, kCsGtile}};
  if ((rc = take_scratch(dev, kCsRedo, redo, n * 4ull + 4)) ||
      (rc = take_scratch(dev, kCsCtr, ctr, (1 + kMaxLines) * kMaxStride * 4)))
    return rc;
  // counters (k_clean_pairs; [3]: pass 2's error bits, [6], [7]: its lists), then the maxima's lines
  uint32_t *cnt = ctr.as<uint32_t>();
  HSDL_HIP(hipMemsetAsync(cnt, 0, (1 + kMaxLines) * kMaxStride * 4, st));
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, idx->device);
  const int grid = std::max(1, cus * 8);
  const unsigned long long *off = idx->off.as<unsigned long long>();
  const unsigned long long *lab = idx->lab.as<unsigned long long>();
  // label pairs, or tiles for long lists (tuning knob HSDL_CLEAN_PAIRS: 0
  // never pairs, 2 always; HSDL_CLEAN_HOP_SORT=0: tiles over the index's own
  // order, no hop-ordered copy)
  const bool hop_sort = env_u32("HSDL_CLEAN_HOP_SORT", 1, 0, 1);
  const uint32_t form = hop_sort ? env_u32("HSDL_CLEAN_PAIRS", 1, 0, 2) : 0u;
  bool pairs = form == 2 || (form == 1 && n >= kPairLists && idx->total <= kPairMean * n);
  const uint64_t hop_bytes = (uint64_t)n * idx->K * 4;
  // The hop-ordered copy and what belongs to it only save time: where the device has
  // no room for them, or for what comes after them, the clean goes on without.
  auto drop_copy = [&] {
    (void)hipStreamSynchronize(st);
    for (DevBuf *b : {&srt, &hcnt, &mins, &longs}) b->release();
  };
  // (the lists that the pairs leave to the tiles stand where the lengths will)
  if (pairs && (take_scratch(dev, kCsLongs, longs, n * 4ull + 4) ||
                take_scratch(dev, kCsNewLen, new_len, n * 4ull) ||
                take_scratch(dev, kCsMins, mins, hop_bytes) ||
                take_scratch(dev, kCsHcnt, hcnt, hop_bytes))) {
    drop_copy();
    new_len.release();
    pairs = false;
  }
  hipLaunchKernelGGL(k_clean_min, dim3(grid), dim3(256), 0, st, n, (uint32_t)idx->K, off, lab,
                     pairs ? mins.as<uint32_t>() : nullptr, cnt + kMaxStride);
  HSDL_HIP(hipGetLastError());
  uint32_t lines[kMaxLines * kMaxStride], mx[2] = {0, 0};
  HSDL_HIP(hipMemcpyAsync(lines, cnt + kMaxStride, sizeof(lines), hipMemcpyDeviceToHost, st));
  HSDL_HIP(hipStreamSynchronize(st));
  for (uint32_t x = 0; x < kMaxLines; ++x)
    for (int y = 0; y < 2; ++y) mx[y] = std::max(mx[y], lines[x * kMaxStride + y]);
  // 32-bit copies of the labels when hub, hop and distance fit one word
  // (tuning knob HSDL_STREAM32=0: 8-byte ones)
  uint32_t hub_bits = 1, hop_bits = 1, dist_bits = 1;
  while ((1ull << hub_bits) <= (uint64_t)(n ? n - 1 : 0)) ++hub_bits;
  while ((1ull << hop_bits) <= (uint64_t)idx->K) ++hop_bits;
  while ((1ull << dist_bits) <= (uint64_t)mx[1]) ++dist_bits;
  const bool use32 =
      env_u32("HSDL_STREAM32", 1, 0, 1) && hub_bits + hop_bits + dist_bits <= 32;
  uint64_t width = use32 ? 4 : 8;
  const uint64_t t_kern = now_ns();
  // k_clean_tile over `cnt` vertices (those of `list`, if any), streaming the hop-
  // ordered 32-bit copy of all labels, or the index
  auto tiles = [&](uint32_t count, const uint32_t *list, bool copy) -> int {
    const uint32_t K1 = (uint32_t)idx->K + 1;
    const bool small_vals = mx[1] < 0xFFFFu;
    // indexed LDS tiles need hub << kIdxBits to fit a word (tuning knob
    // HSDL_CLEAN_INDEXED=0: per-slot values only)
    const uint32_t indexed =
        (uint64_t)n <= (1ull << (32 - kIdxBits)) ? env_u32("HSDL_CLEAN_INDEXED", 1, 0, 1) : 0u;
    const uint32_t slot_bytes = 4 + K1 * (small_vals ? 2 : 4);
    // tuning knob HSDL_CLEAN_LDS_SLOTS caps the LDS tile (small values send
    // every vertex to the global arena)
    uint32_t lds_slots = (kTileLdsBytes - 16) / slot_bytes;
    lds_slots = env_u32("HSDL_CLEAN_LDS_SLOTS", lds_slots, 1, lds_slots);
    const size_t lds_bytes = (size_t)lds_slots * slot_bytes + 16;
    const int tgrid = std::max(1, cus * 2);
    // tuning knob HSDL_CLEAN_WINDOW: labels of L(v) per wave work unit
    const uint32_t win = env_u32("HSDL_CLEAN_WINDOW", kTileWindow, 1, kMaxWindow);
    const uint32_t gcap = tile_cap_for(mx[0]);
    const uint64_t gwords =
        small_vals ? tile_words<uint16_t>(gcap, K1) : tile_words<uint32_t>(gcap, K1);
    if ((rc = take_scratch(dev, kCsGtile, gtile, (uint64_t)tgrid * gwords * 4))) {
      if (!srt.p) return rc;
      drop_copy();
      copy = false;
      width = 8;
      if ((rc = take_scratch(dev, kCsGtile, gtile, (uint64_t)tgrid * gwords * 4))) return rc;
    }
    auto launch = [&](auto kern, auto str) {
      hipLaunchKernelGGL(kern, dim3(tgrid), dim3(kTileThreads), lds_bytes, st, count, list,
                         (uint32_t)idx->K, off, lab, str, redo.as<uint32_t>(), cnt, lds_slots,
                         gtile.as<uint32_t>(), gwords, win, indexed);
    };
    const Stream32 s32{srt.as<uint32_t>(), hop_bits, dist_bits, hcnt.as<uint32_t>(),
                       (uint32_t)idx->K};
    const Stream64 s64{lab};
    if (small_vals) {
      if (copy) launch(k_clean_tile<uint16_t, Stream32>, s32);
      else launch(k_clean_tile<uint16_t, Stream64>, s64);
    } else {
      if (copy) launch(k_clean_tile<uint32_t, Stream32>, s32);
      else launch(k_clean_tile<uint32_t, Stream64>, s64);
    }
    HSDL_HIP(hipGetLastError());
    return HSDL_OK;
  };
  uint32_t hc[9] = {};  // the counters (k_clean_pairs)
  auto counters = [&]() -> int {
    HSDL_HIP(hipMemcpyAsync(hc, ctr.p, sizeof(hc), hipMemcpyDeviceToHost, st));
    HSDL_HIP(hipStreamSynchronize(st));
    return HSDL_OK;
  };
  // The hop-ordered copy of the pairs holds a slice of the vertices: all of them up to
  // kSliceBytes (tuning knob HSDL_CLEAN_SLICE: labels), fewer when there is no room
  // for it, at least the longest list.
  constexpr uint64_t kSliceBytes = 2ull << 30;
  constexpr uint64_t kPad = 64;  // labels read past a list's end (masked)
  uint64_t cap = std::min<uint64_t>(idx->total, kSliceBytes / width);
  cap = std::max<uint64_t>({std::min<uint64_t>(cap, env_u32("HSDL_CLEAN_SLICE", 0xFFFFFFFFu, 1,
                                                           0xFFFFFFFFu)),
                            mx[0], 1});
  while (pairs && take_scratch(dev, kCsSrt, srt, (cap + kPad) * width)) {
    if (cap <= mx[0]) {
      drop_copy();
      pairs = false;
    }
    cap = std::max<uint64_t>(cap / 2, mx[0]);
  }
  if (pairs) {
    std::vector<uint64_t> hoff;
    if (idx->total > cap) {
      hoff.resize(n + 1ull);
      HSDL_HIP(hipMemcpy(hoff.data(), off, (n + 1ull) * 8, hipMemcpyDeviceToHost));
    }
    auto pass1 = [&](auto f) -> int {
      using F = decltype(f);
      using T = typename F::T;
      for (uint32_t v0 = 0; v0 < n;) {
        uint32_t v1 = n;
        if (!hoff.empty()) {
          const uint64_t end = hoff[v0] + cap;
          v1 = (uint32_t)(std::upper_bound(hoff.begin() + v0, hoff.end(), end) - hoff.begin()) - 1;
        }
        hipLaunchKernelGGL(k_clean_sort<F>, dim3(grid), dim3(256), 0, st, f, v0, v1,
                           (uint32_t)idx->K, off, lab, srt.as<T>(), hcnt.as<uint32_t>());
        HSDL_HIP(hipGetLastError());
        HSDL_HIP(hipMemsetAsync(cnt + 1, 0, 8, st));
        hipLaunchKernelGGL((k_clean_pairs<F, false>), dim3(grid), dim3(256), 0, st, f, v0, v1,
                           (uint32_t)idx->K, off, lab, srt.as<T>(), hcnt.as<uint32_t>(),
                           mins.as<uint32_t>(), redo.as<uint32_t>(), longs.as<uint32_t>(),
                           new_len.as<uint32_t>(), cnt);
        HSDL_HIP(hipGetLastError());
        if (mx[0] > kCleanLong) {
          HSDL_HIP(hipMemsetAsync(cnt + 2, 0, 4, st));
          hipLaunchKernelGGL((k_clean_pairs<F, true>), dim3(grid), dim3(256), 0, st, f, v0, v1,
                             (uint32_t)idx->K, off, lab, srt.as<T>(), hcnt.as<uint32_t>(),
                             mins.as<uint32_t>(), redo.as<uint32_t>(), longs.as<uint32_t>(),
                             new_len.as<uint32_t>(), cnt);
          HSDL_HIP(hipGetLastError());
        }
        v0 = v1;
      }
      return HSDL_OK;
    };
    if (idx->total && (rc = use32 ? pass1(Pair32{hop_bits, dist_bits}) : pass1(Pair64{})))
      return rc;
    if ((rc = counters())) return rc;
    if (hc[8]) {
      HSDL_HIP(hipMemsetAsync(cnt + 2, 0, 4, st));
      if ((rc = tiles(hc[8], new_len.as<uint32_t>(), use32 && hoff.empty())) || (rc = counters()))
        return rc;
    }
  } else {
    // the heads' lists are streamed from a hop-ordered 32-bit copy of all
    // labels, or from the index when fields or memory do not allow it
    const bool copy = use32 && hop_sort &&
                      take_scratch(dev, kCsHcnt, hcnt, hop_bytes) == HSDL_OK &&
                      take_scratch(dev, kCsSrt, srt, idx->total * 4) == HSDL_OK;
    if (copy) {
      hipLaunchKernelGGL(k_clean_sort<Pair32>, dim3(grid), dim3(256), 0, st,
                         Pair32{hop_bits, dist_bits}, 0u, n, (uint32_t)idx->K, off, lab,
                         srt.as<uint32_t>(), hcnt.as<uint32_t>());
      HSDL_HIP(hipGetLastError());
    } else {
      width = 8;
    }
    if ((rc = tiles(n, nullptr, copy)) || (rc = counters())) return rc;
  }
  const uint64_t t_passes = now_ns();
  // nothing falls: the index stays as it is
  if (hc[0]) {
    // (the first pass has ended: its buffers make room)
    auto with_room = [&](auto &&alloc) -> int {
      if (alloc() == HSDL_OK) return HSDL_OK;
      drop_copy();
      gtile.release();
      return alloc();
    };
    auto take = [&](int id, DevBuf &b, uint64_t bytes) {
      return with_room([&] { return take_scratch(dev, id, b, bytes); });
    };
    if ((rc = take(kCsKeep, keep, std::max<uint64_t>(idx->total, 1))) ||
        (!new_len.p && (rc = take(kCsNewLen, new_len, n * 4ull))) ||
        (rc = take(kCsOff, noff, (n + 1ull) * 8)))
      return rc;
    HSDL_HIP(hipMemsetAsync(keep.p, 1, idx->total, st));
    hipLaunchKernelGGL(k_clean_keep_all, dim3(grid), dim3(256), 0, st, n, off,
                       new_len.as<uint32_t>());
    HSDL_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_clean_seq<false>, dim3(cus * 3), dim3(kSeqThreads), 0, st,
                       (uint32_t)idx->K, off, lab, keep.as<uint8_t>(), new_len.as<uint32_t>(),
                       redo.as<uint32_t>(), cnt, cnt + 6, cnt + 3, nullptr, 0u);
    HSDL_HIP(hipGetLastError());
    DevBuf long_bits;
    if (mx[0] > kSeqBits) {
      // vertices with more labels than an LDS bit set holds: bits in a global
      // slice per workgroup (few workgroups: such vertices are rare)
      const uint32_t lgrid = 64;
      const uint32_t words = (mx[0] + 31) / 32;
      if ((rc = with_room([&] { return long_bits.alloc((uint64_t)lgrid * 2 * words * 4); })))
        return rc;
      hipLaunchKernelGGL(k_clean_seq<true>, dim3(lgrid), dim3(kSeqThreads), 0, st,
                         (uint32_t)idx->K, off, lab, keep.as<uint8_t>(), new_len.as<uint32_t>(),
                         redo.as<uint32_t>(), cnt, cnt + 7, cnt + 3, long_bits.as<uint32_t>(),
                         words);
      HSDL_HIP(hipGetLastError());
    }
    uint32_t bad = 0;
    HSDL_HIP(hipMemcpyAsync(&bad, cnt + 3, 4, hipMemcpyDeviceToHost, st));
    HSDL_HIP(hipStreamSynchronize(st));
    if (bad & 2u) return fail(HSDL_EINVAL, "a vertex holds more than 32 labels of one hub");
    if (bad) return fail(HSDL_EDEVICE, "clean: keep-bit scratch smaller than a list");
    if ((rc = scan_counts_u32(new_len.as<uint32_t>(), noff.as<uint64_t>(), n, st))) return rc;
    uint64_t total = 0;
    HSDL_HIP(hipMemcpy(&total, noff.as<uint64_t>() + n, 8, hipMemcpyDeviceToHost));
    if ((rc = take(kCsLab, nlab, std::max<uint64_t>(total, 1) * 8))) return rc;
    DevBuf npar;
    if (idx->has_parents &&
        (rc = with_room([&] { return npar.alloc(std::max<uint64_t>(total, 1) * 4); })))
      return rc;
    hipLaunchKernelGGL(k_compact, dim3(grid), dim3(256), 0, st, n, off, lab, keep.as<uint8_t>(),
                       noff.as<unsigned long long>(), nlab.as<unsigned long long>(),
                       idx->has_parents ? idx->par.as<uint32_t>() : nullptr,
                       idx->has_parents ? npar.as<uint32_t>() : nullptr);
    HSDL_HIP(hipGetLastError());
    HSDL_HIP(hipStreamSynchronize(st));
    // the replaced arrays are kept for the next clean's new ones
    std::swap(idx->off, noff);
    std::swap(idx->lab, nlab);
    idx->lab32.release();
    idx->q32.store(0, std::memory_order_release);
    give_scratch(dev, kCsOff, noff);
    give_scratch(dev, kCsLab, nlab);
    if (idx->has_parents) idx->par = std::move(npar);
    idx->total = total;
  }
  give.idle = true;
  idx->cleaned = true;
  idx->stats.labels_cleaned = idx->total;
  idx->stats.clean_passes = hc[0] ? 2 : 1;
  idx->stats.clean_seq_vertices = hc[0];
  idx->stats.clean_label_reads = (uint64_t)hc[4] | ((uint64_t)hc[5] << 32);
  idx->stats.clean_label_bytes = (uint32_t)width;
  const uint64_t t_end = now_ns();
  idx->stats.t_clean_s = (t_end - t0) * 1e-9;
  if (getenv("HSDL_VERBOSE"))
    fprintf(stderr, "[hsdl] clean: %.3f s set-up, %.3f s pass 1 (%u lists left to tiles), "
            "%.3f s pass 2 and compaction\n",
            (t_kern - t0) * 1e-9, (t_passes - t_kern) * 1e-9, hc[8], (t_end - t_passes) * 1e-9);
  return HSDL_OK;
}

}  // namespace hsdl

static int clean_body(hsdl_index *idx) {
  if (!idx) return hsdl::fail(HSDL_EINVAL, "null index");
  return hsdl::clean_index(idx);
}

extern "C" int hsdl_clean(hsdl_index *idx) {
  return hsdl::guarded([&] { return clean_body(idx); });
}

static int release_scratch_body(int32_t device) {
  int was = -1;
  (void)hipGetDevice(&was);
  hsdl::release_stages(device);
  if (was >= 0) (void)hipSetDevice(was);
  std::lock_guard<std::mutex> lk(hsdl::g_clean_scratch_mu);
  int cur = -1;
  (void)hipGetDevice(&cur);
  for (int d = 0; d < hsdl::kCsDevices; ++d) {
    if (device >= 0 && d != device) continue;
    hsdl::CleanScratch &c = hsdl::g_clean_scratch[d];
    bool any = false;
    for (int i = 0; i < hsdl::kCsCount; ++i) any |= c.p[i] != nullptr;
    if (!any) continue;
    (void)hipSetDevice(d);
    for (int i = 0; i < hsdl::kCsCount; ++i) {
      if (c.p[i]) (void)hipFree(c.p[i]);
      c.p[i] = nullptr;
      c.bytes[i] = 0;
    }
  }
  if (cur >= 0) (void)hipSetDevice(cur);
  return HSDL_OK;
}

extern "C" int hsdl_release_scratch(int32_t device) {
  return hsdl::guarded([&] { return release_scratch_body(device); });
}
