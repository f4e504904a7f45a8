// query.hip -- batched (s,t,k) hop-bounded distance queries on gfx950.
//
// Semantics of hop_constrained_extract_distance
// (CPU_HopHL/include/HBPLL/hop_constrained_two_hop_labels.h:144-222):
//   k < 0 -> INT32_MAX; s == t -> 0; k == 0 -> INT32_MAX; otherwise
//   min{ d1 + d2 : (w,h1,d1) in L(s), (w,h2,d2) in L(t), h1 + h2 <= k }
//   or INT32_MAX when no pair qualifies.
// The reference's GPU query (Query_mdnd/src/gpu_query.cu:5-177) launches three
// kernels per query; here one launch answers a whole batch.
//
// A wavefront per query, with its own slice of LDS and no barriers, in one of
// two forms.  A wave takes up to 64 consecutive queries of the batch at a time,
// as many as leave every resident wave some: their requests are one coalesced
// load and their answers one store, which counts where the server's requests
// lie in host memory.
//
// k_query32 reads the index's 32-bit query copy, which keeps every list by hop
// with prefix counts.  With a and b the endpoints (a's list the shorter one)
// and c = k / 2, a pair falls in one of
//   h1 in 1..c,     h2 in 1..k-1:    a's labels of hop 1..c are hashed by hub,
//                                    b's labels of hop 1..k-1 probe them;
//   h1 in c+1..k-1, h2 in 1..k-1-c:  b's labels of hop 1..k-1-c are hashed,
//                                    a's labels of hop c+1..k-1 probe them;
//   h1 = 0 or h2 = 0:                a label of hub a in L(b), or of hub b in
//                                    L(a), with the other's self label.
// Most labels have hops 2 and 3, so a query with k < K reads a part of its
// lists and hashes a smaller one.  Labels of hop k matter only for hub a or b,
// which ranks above the list's vertex: only the lower-ranked endpoint's list is
// read that far, unless the index holds hubs ranked below their vertex
// (imported label sets may).  A query with a part of more labels than half the
// table reads the 8-byte labels as k_query64 does; hashing it in pieces streamed
// the other list once per piece (20,000 queries between lists of 5,000 labels 1.37
// ms, now 0.52).  What binds is instructions (a probe about 15
// for 64 labels, a turn of its chain 10): 2^22 queries of an R-MAT 262,144
// index at K = 5 (672 labels per list, k uniform in 1..5) take 5.24 ms, 800 M
// q/s; a workgroup of four waves per query, with both whole lists in registers
// and LDS, took 19.2 ms.
//
// k_query64 reads the index's 8-byte labels, in (hub, hop, dist) order, where
// there is no copy (fields wider than 32 bits, no memory, none made yet).  The
// longer list is staged in LDS in pieces of 512 labels, and the shorter one's
// labels whose hubs lie in the piece's range search it.  The same
// 2^22 queries without the copy: 23.7 -> 10.9 ms; 100,003 queries on a 384 x 401
// grid's index (63 labels per list, K = 8) from host arrays: 0.51 -> 0.18 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "device.hpp"

namespace hsdl {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kQThreads = 256;  // four queries
constexpr uint32_t kQWaves = kQThreads / kWave;

// The query copy's labels: hub << (hop_bits + dist_bits) | hop << dist_bits |
// dist.  No label of hop >= 1 is 0.
struct Lab32 {
  uint32_t db, hsh, hmask, dmask;  // dist bits, hop + dist bits, field masks
  __device__ uint32_t hub(uint32_t l) const { return l >> hsh; }
  __device__ uint32_t hop(uint32_t l) const { return (l >> db) & hmask; }
  __device__ uint32_t dist(uint32_t l) const { return l & dmask; }
};

// Queries a wave takes at a time.
struct QChunk {
  uint32_t per;
  __device__ QChunk(uint64_t nq, uint64_t waves)
      : per((uint32_t)min<uint64_t>(kWave, (nq + waves - 1) / waves)) {}
};

// 8-byte labels: pieces of the longer list B in LDS, searched by the shorter
// list A's labels.  Both are hub-sorted, so a chunk of A whose hubs lie below
// the piece is never read again; a run of B cut by a piece's end is found in
// both pieces.
// kN threads' work: a wave's, or a workgroup's (a piece of 512 labels per wave,
// the waves taking chunks of A in turn).  Returns the least distance of (s, t, k),
// k > 0, s != t, over this lane's pairs.
constexpr uint32_t kQPiece = 512;  // labels, 4 KB per wave
// Where B is far the longer, A's labels search it in memory: 100,000 queries of a
// list of 20 labels and one of 16,000 (60,000) 0.87 -> 0.11 ms (2.6 -> 0.12).  The
// search is a chain of a dozen loads: between lists of up to 8,192 labels that lie
// in HBM (R-MAT 2^20 vertices, K = 5) it loses to the pieces, 9.2 against 8.4 ms.
constexpr uint32_t kQSearchLen = 8192;
constexpr uint32_t kQSearchRatio = 64;
__device__ inline bool searched(uint32_t alen, uint32_t blen) {
  return blen > kQSearchLen && (uint64_t)alen * kQSearchRatio <= blen;
}
template <uint32_t kN>
__device__ inline uint32_t join64(const unsigned long long *__restrict__ off,
                                  const unsigned long long *__restrict__ lab, uint32_t s,
                                  uint32_t t, uint32_t kk, lds_ptr<unsigned long long> P) {
  constexpr bool kTeam = kN > kWave;
  constexpr uint32_t kPiece = kN / kWave * kQPiece;
  const uint32_t lane = (uint32_t)lane_id(), id = kTeam ? threadIdx.x : lane;
  auto sync = [] {
    if constexpr (kTeam)
      __syncthreads();
    else
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  unsigned long long abeg = off[s], bbeg = off[t];
  uint32_t alen = (uint32_t)(off[s + 1] - abeg), blen = (uint32_t)(off[t + 1] - bbeg);
  if (alen > blen) {
    const unsigned long long x = abeg; abeg = bbeg; bbeg = x;
    const uint32_t l = alen; alen = blen; blen = l;
  }
  const unsigned long long *A = lab + abeg, *B = lab + bbeg;
  uint32_t best = kInf32;
  // this wave's chunks of A below j0 are done
  uint32_t j0 = kTeam ? __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) * kWave : 0u;
  if (searched(alen, blen)) {
    for (; j0 < alen; j0 += kN) {
      const unsigned long long a = A[min(j0 + lane, alen - 1)];
      const uint32_t w = label_hub(a), h1 = label_hop(a);
      if (h1 > kk) continue;
      uint32_t lo = 0, hi = blen;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (label_hub(B[mid]) < w) lo = mid + 1; else hi = mid;
      }
      for (; lo < blen; ++lo) {  // <= K + 1 labels, hops ascending
        const unsigned long long l = B[lo];
        if (label_hub(l) != w || h1 + label_hop(l) > kk) break;
        best = min(best, label_dist(a) + label_dist(l));
      }
    }
    return best;
  }
  for (uint32_t p0 = 0; p0 < blen && (kTeam || j0 < alen); p0 += kPiece) {
    const uint32_t m = min(kPiece, blen - p0);
    for (uint32_t i = id; i < m; i += 4 * kN) {
      unsigned long long l[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) l[u] = B[p0 + min(i + u * kN, m - 1)];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        if (i + u * kN < m) P[i + u * kN] = l[u];
    }
    sync();
    const uint32_t lo_hub = label_hub(P[0]), hi_hub = label_hub(P[m - 1]);
    for (uint32_t j = j0; j < alen; j += kN) {
      const unsigned long long a = A[min(j + lane, alen - 1)];
      const uint32_t w = label_hub(a), h1 = label_hop(a);
      if (__builtin_amdgcn_readlane(w, 0) > hi_hub) break;
      if (__builtin_amdgcn_readlane(w, kWave - 1) < lo_hub) {
        j0 = j + kN;
        continue;
      }
      if (w < lo_hub || w > hi_hub || h1 > kk) continue;
      // first label of the piece with hub >= w (there is one)
      uint32_t lo = 0, hi = m - 1;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (label_hub(P[mid]) < w) lo = mid + 1; else hi = mid;
      }
      for (uint32_t x = lo; x < m; ++x) {  // <= K + 1 labels, hops ascending
        const unsigned long long l = P[x];
        if (label_hub(l) != w || h1 + label_hop(l) > kk) break;
        best = min(best, label_dist(a) + label_dist(l));
      }
    }
    sync();
  }
  return best;
}

// LDS words of a wave of the query copy's kernels: its table, or a piece of 8-byte
// labels.
__host__ __device__ inline uint32_t slice_words(uint32_t slots) {
  return slots > 2 * kQPiece ? slots : 2 * kQPiece;
}

// The least distance of (s, t, k), k > 0, s != t, over this lane's pairs
// (kInf32: none).  kN threads' work: a wave's, or a workgroup's in step.
// hcnt[v * K + x], x < K: labels of v of hop <= x.  below: the index holds hubs
// ranked below their vertex.  T: slice_words per wave, a table of `slots`, a power
// of two.  lab64: the 8-byte labels.
template <uint32_t kN>
__device__ inline uint32_t join32(const Lab32 &fmt, uint32_t K,
                                  const unsigned long long *__restrict__ off,
                                  const uint32_t *__restrict__ lab,
                                  const uint32_t *__restrict__ hcnt, uint32_t below, uint32_t s,
                                  uint32_t t, int k, lds_ptr<uint32_t> T, uint32_t slots,
                                  const unsigned long long *__restrict__ lab64) {
  constexpr bool kTeam = kN > kWave;
  const uint32_t id = kTeam ? threadIdx.x : (uint32_t)lane_id();
  auto sync = [] {
    if constexpr (kTeam)
      __syncthreads();
    else
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  uint32_t a = s, b = t;
  unsigned long long abeg = off[s], bbeg = off[t];
  uint32_t alen = (uint32_t)(off[s + 1] - abeg), blen = (uint32_t)(off[t + 1] - bbeg);
  if (alen > blen) {
    const unsigned long long x = abeg; abeg = bbeg; bbeg = x;
    const uint32_t l = alen; alen = blen; blen = l;
    a = t;
    b = s;
  }
  const uint32_t *A = lab + abeg, *B = lab + bbeg;
  const uint32_t kk = (uint32_t)k, c = kk >> 1;
  // labels of v of hop <= x
  auto upto = [&](uint32_t v, uint32_t len, uint32_t x) {
    return x < K ? hcnt[(uint64_t)v * K + x] : len;
  };
  const uint32_t a0 = upto(a, alen, 0), b0 = upto(b, blen, 0);  // self labels
  const uint32_t ac = upto(a, alen, c), bc = upto(b, blen, kk - 1 - c);
  const uint32_t a1 = upto(a, alen, kk - 1), b1 = upto(b, blen, kk - 1);
  const uint32_t ak = upto(a, alen, kk), bk = upto(b, blen, kk);
  // a part that outgrows the table, or a list that is searched
  if (__builtin_expect(max(ac - a0, bc - b0) > slots / 2 || searched(alen, blen), 0))
    return join64<kN>(off, lab64, s, t, kk, (lds_ptr<unsigned long long>)T);
  uint32_t best = kInf32;       // pairs of hops >= 1
  uint32_t at_a = kInf32, at_b = kInf32;  // labels of hub a in L(b), of b in L(a)

  // Labels [beg, end) of L, four steps' loads at a time; use(l, own) sees every
  // label (a lane past the end a copy of the last one, own = false).
  auto walk = [&](const uint32_t *L, uint32_t beg, uint32_t end, auto &&use) {
    for (uint32_t j = beg; j < end; j += 4 * kN) {
      uint32_t l[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) l[u] = L[min(j + u * kN + id, end - 1)];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        if (j + u * kN < end) use(l[u], j + u * kN + id < end);
    }
  };
  auto endpoint = [&](uint32_t l, uint32_t other, uint32_t &at) {
    if (fmt.hub(l) == other) at = min(at, fmt.dist(l));
  };
  // hashes X[xb, xe), probes with Y[yb, ye)
  auto join = [&](const uint32_t *X, uint32_t xb, uint32_t xe, const uint32_t *Y, uint32_t yb,
                  uint32_t ye) {
    if (xb >= xe || yb >= ye) return;
    // at most half the table; a quarter where it has room
    const uint32_t cap = min(slots, 1u << (32 - __builtin_clz(max(64u, 4u * (xe - xb)) - 1)));
    for (uint32_t i = id; i < cap * 4 / 16; i += kN) ((lds_ptr<u32x4>)T)[i] = u32x4{0, 0, 0, 0};
    sync();
    walk(X, xb, xe, [&](uint32_t l, bool own) {
      if (!own) return;
      uint32_t slot = hash_slot(fmt.hub(l), cap);
      while (atomicCAS((uint32_t *)&T[slot], 0u, l) != 0u) slot = (slot + 1) & (cap - 1);
    });
    sync();
    walk(Y, yb, ye, [&](uint32_t l, bool) {
      const uint32_t w = fmt.hub(l), h = fmt.hop(l), d = fmt.dist(l);
      uint32_t slot = hash_slot(w, cap);
      uint32_t x = T[slot];
      while (x != 0) {
        if (fmt.hub(x) == w && fmt.hop(x) + h <= kk) best = min(best, d + fmt.dist(x));
        slot = (slot + 1) & (cap - 1);
        x = T[slot];
      }
    });
    sync();
  };
  if (below || b > a) walk(B, b0, bk, [&](uint32_t l, bool) { endpoint(l, a, at_a); });
  if (below || a > b) walk(A, a0, ak, [&](uint32_t l, bool) { endpoint(l, b, at_b); });
  join(A, a0, ac, B, b0, b1);
  join(B, b0, bc, A, ac, a1);
  if (a0) best = min(best, at_a);
  if (b0) best = min(best, at_b);
  return best;
}

// A wave per query.  slots: table slots per wave.
__global__ void __launch_bounds__(kQThreads) __attribute__((amdgpu_waves_per_eu(8)))
k_query32(Lab32 fmt, uint32_t n, uint32_t K, const unsigned long long *__restrict__ off,
          const uint32_t *__restrict__ lab, const uint32_t *__restrict__ hcnt, uint32_t below,
          uint64_t nq, const uint32_t *__restrict__ qs, const uint32_t *__restrict__ qt,
          const int8_t *__restrict__ qk, int32_t *out, uint32_t slots,
          const unsigned long long *__restrict__ lab64) {
  extern __shared__ uint4 qlds[];  // 16-byte stores clear the tables
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  lds_ptr<uint32_t> T =
      (lds_ptr<uint32_t>)(reinterpret_cast<uint32_t *>(qlds) + wib * slice_words(slots));
  const uint64_t waves = (uint64_t)gridDim.x * kQWaves;
  const QChunk ch(nq, waves);
  for (uint64_t q0 = ((uint64_t)blockIdx.x * kQWaves + wib) * ch.per; q0 < nq;
       q0 += waves * ch.per) {
    // lane i: request q0 + i, then its answer
    const uint32_t cnt = (uint32_t)min<uint64_t>(ch.per, nq - q0);
    const bool mine = lane < cnt;
    const uint32_t vs = mine ? qs[q0 + lane] : 0u, vt = mine ? qt[q0 + lane] : 0u;
    const int vk = mine ? qk[q0 + lane] : 0;
    int32_t ans = vk >= 0 && vs == vt && vs < n ? 0 : INT32_MAX;
    // the others need a join
    for (unsigned long long todo = __ballot(vk > 0 && vs < n && vt < n && vs != vt); todo;
         todo &= todo - 1) {
      const int qi = __ffsll((long long)todo) - 1;
      const uint32_t best = wave_min_u32(
          join32<kWave>(fmt, K, off, lab, hcnt, below, __builtin_amdgcn_readlane(vs, qi),
                        __builtin_amdgcn_readlane(vt, qi), __builtin_amdgcn_readlane(vk, qi), T,
                        slots, lab64));
      if ((int)lane == qi) ans = best == kInf32 ? INT32_MAX : (int32_t)best;
    }
    if (mine) out[q0 + lane] = ans;
  }
}

// A workgroup per query, for calls of few queries (use_team): the longest lists'
// queries decide when such a call ends, and its waves would idle beside them.  The
// workgroup takes consecutive queries, as many as leave every resident one some:
// the first wave loads their requests together for all waves, and the answers are
// stored together.  (Each wave loading each request by itself made three reads of
// host memory per wave of a server's requests: R-MAT 262,144 at 30 M requests/s
// 38 us at the median against 34.)
// join(s, t, k) is called by all threads of the workgroup.
template <uint32_t kN, class J>
__device__ inline void team_queries(uint32_t n, uint64_t nq, const uint32_t *__restrict__ qs,
                                    const uint32_t *__restrict__ qt,
                                    const int8_t *__restrict__ qk, int32_t *out, J &&join) {
  __shared__ uint32_t least[kN / kWave], rs[kWave], rt[kWave];
  __shared__ int rk[kWave];
  const uint32_t tid = threadIdx.x;
  const uint32_t wib = __builtin_amdgcn_readfirstlane(tid / kWave);
  const QChunk ch(nq, gridDim.x);
  for (uint64_t q0 = blockIdx.x * (uint64_t)ch.per; q0 < nq; q0 += gridDim.x * (uint64_t)ch.per) {
    const uint32_t cnt = (uint32_t)min<uint64_t>(ch.per, nq - q0);
    if (tid < cnt) {
      rs[tid] = qs[q0 + tid];
      rt[tid] = qt[q0 + tid];
      rk[tid] = qk[q0 + tid];
    }
    __syncthreads();
    int32_t ans = 0;  // thread i: query q0 + i's
    for (uint32_t i = 0; i < cnt; ++i) {
      const uint32_t s = __builtin_amdgcn_readfirstlane(rs[i]);
      const uint32_t t = __builtin_amdgcn_readfirstlane(rt[i]);
      const int k = __builtin_amdgcn_readfirstlane(rk[i]);
      uint32_t best = kInf32;
      if (k > 0 && s < n && t < n && s != t)  // the same for every thread
        best = wave_min_u32(join(s, t, k));
      if (lane_id() == 0) least[wib] = best;
      __syncthreads();
#pragma unroll
      for (uint32_t w = 0; w < kN / kWave; ++w) best = min(best, least[w]);
      if (tid == i) ans = k >= 0 && s == t && s < n ? 0 : best == kInf32 ? INT32_MAX : (int32_t)best;
      __syncthreads();  // `least`, the requests and the join's LDS are the next query's
    }
    if (tid < cnt) out[q0 + tid] = ans;
  }
}

// slots: table slots of the workgroup.
template <uint32_t kN>
__global__ void __launch_bounds__(kN) __attribute__((amdgpu_waves_per_eu(8)))
k_query32_team(Lab32 fmt, uint32_t n, uint32_t K, const unsigned long long *__restrict__ off,
               const uint32_t *__restrict__ lab, const uint32_t *__restrict__ hcnt,
               uint32_t below, uint64_t nq, const uint32_t *__restrict__ qs,
               const uint32_t *__restrict__ qt, const int8_t *__restrict__ qk, int32_t *out,
               uint32_t slots, const unsigned long long *__restrict__ lab64) {
  extern __shared__ uint4 qlds[];
  team_queries<kN>(n, nq, qs, qt, qk, out, [&](uint32_t s, uint32_t t, int k) {
    return join32<kN>(fmt, K, off, lab, hcnt, below, s, t, k,
                      (lds_ptr<uint32_t>)reinterpret_cast<uint32_t *>(qlds), slots, lab64);
  });
}

__global__ void __launch_bounds__(kQThreads) __attribute__((amdgpu_waves_per_eu(8)))
k_query64(uint32_t n, const unsigned long long *__restrict__ off,
          const unsigned long long *__restrict__ lab, uint64_t nq,
          const uint32_t *__restrict__ qs, const uint32_t *__restrict__ qt,
          const int8_t *__restrict__ qk, int32_t *out) {
  __shared__ unsigned long long stage[kQWaves][kQPiece];
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t waves = (uint64_t)gridDim.x * kQWaves;
  const QChunk ch(nq, waves);
  for (uint64_t q0 = ((uint64_t)blockIdx.x * kQWaves + wib) * ch.per; q0 < nq;
       q0 += waves * ch.per) {
    // lane i: request q0 + i, then its answer
    const uint32_t cnt = (uint32_t)min<uint64_t>(ch.per, nq - q0);
    const bool mine = lane < cnt;
    const uint32_t vs = mine ? qs[q0 + lane] : 0u, vt = mine ? qt[q0 + lane] : 0u;
    const int vk = mine ? qk[q0 + lane] : 0;
    int32_t ans = vk >= 0 && vs == vt && vs < n ? 0 : INT32_MAX;
    // the others need a join
    for (unsigned long long todo = __ballot(vk > 0 && vs < n && vt < n && vs != vt); todo;
         todo &= todo - 1) {
      const int qi = __ffsll((long long)todo) - 1;
      const uint32_t best = wave_min_u32(join64<kWave>(
          off, lab, __builtin_amdgcn_readlane(vs, qi), __builtin_amdgcn_readlane(vt, qi),
          (uint32_t)__builtin_amdgcn_readlane(vk, qi), (lds_ptr<unsigned long long>)stage[wib]));
      if ((int)lane == qi) ans = best == kInf32 ? INT32_MAX : (int32_t)best;
    }
    if (mine) out[q0 + lane] = ans;
  }
}

template <uint32_t kN>
__global__ void __launch_bounds__(kN) __attribute__((amdgpu_waves_per_eu(8)))
k_query64_team(uint32_t n, const unsigned long long *__restrict__ off,
               const unsigned long long *__restrict__ lab, uint64_t nq,
               const uint32_t *__restrict__ qs, const uint32_t *__restrict__ qt,
               const int8_t *__restrict__ qk, int32_t *out) {
  __shared__ unsigned long long stage[kN / kWave * kQPiece];
  team_queries<kN>(n, nq, qs, qt, qk, out, [&](uint32_t s, uint32_t t, int k) {
    return join64<kN>(off, lab, s, t, (uint32_t)k, (lds_ptr<unsigned long long>)stage);
  });
}

// Workgroups resident at once on a device (the persistent grid), cached per
// kernel and LDS size.
static uint32_t query_grid(int dev, bool copy, size_t lds) {
  struct Cache {
    int dev = -1;
    size_t lds = 0;
    uint32_t grid = 0;
  };
  static std::mutex mu;
  static Cache cache[2];
  std::lock_guard<std::mutex> g(mu);
  Cache &c = cache[copy];
  if (dev == c.dev && lds == c.lds) return c.grid;
  int cus = 0, per_cu = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  const hipError_t e =
      copy ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_query32, kQThreads, lds)
           : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_query64, kQThreads, lds);
  if (e != hipSuccess || per_cu <= 0) per_cu = 4;
  c = Cache{dev, lds, (uint32_t)(cus * per_cu)};
  return c.grid;
}

// The query copy: every list's labels as 32-bit words in hop order (any order
// within a hop) and the prefix counts, a wave per list.  An index's first call waits for
// it.  Lists of up to kPackHeld labels are read once, held in registers while their
// labels are ranked hop by hop, and stored from LDS in whole lines.  First calls on
// R-MAT 262,144 (672 labels per list) 1,275 -> 950 us, on 65,536 at K = 3 / 5 118 / 157 ->
// 98 / 123, against a wave per list that read it twice and stored label by label (a copy
// in the index's own order: 520, 70 and 120).
constexpr uint32_t kPackRegs = 16, kPackHeld = kPackRegs * kWave;
struct PackArgs {
  uint32_t n, K;
  const unsigned long long *off, *lab;
  uint32_t *out, *hcnt;
  uint32_t hsh, db;
  __device__ uint32_t word(unsigned long long l) const {
    return (label_hub(l) << hsh) | (label_hop(l) << db) | label_dist(l);
  }
};
__global__ void __launch_bounds__(kQThreads) k_pack_short(PackArgs a) {
  __shared__ uint32_t sorted[kQWaves][kPackHeld];
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  lds_ptr<uint32_t> T = (lds_ptr<uint32_t>)sorted[wib];
  const uint32_t wave = blockIdx.x * kQWaves + wib, nwaves = gridDim.x * kQWaves;
  // the extents of up to 64 lists together
  const uint32_t per = min((uint32_t)kWave, (a.n + nwaves - 1) / nwaves);
  for (uint64_t v0 = (uint64_t)wave * per; v0 < a.n; v0 += (uint64_t)nwaves * per) {
    const uint32_t cnt = (uint32_t)min<uint64_t>(per, a.n - v0);
    const uint64_t vi = v0 + min(lane, cnt - 1);
    const unsigned long long vb = a.off[vi];
    const uint32_t vlen = (uint32_t)min<uint64_t>(a.off[vi + 1] - vb, kInf32);
    for (uint32_t i = 0; i < cnt; ++i) {
      const uint32_t len = __builtin_amdgcn_readlane(vlen, i);
      if (len > kPackHeld) continue;  // k_pack_long's
      const unsigned long long b =
          ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((uint32_t)(vb >> 32), i) << 32) |
          (uint32_t)__builtin_amdgcn_readlane((uint32_t)vb, i);
      const unsigned long long *L = a.lab + b;
      unsigned long long l[kPackRegs];
      uint32_t p[kPackRegs], dst[kPackRegs];
#pragma unroll
      for (uint32_t r = 0; r < kPackRegs; ++r) {
        l[r] = 0;
        if (r * kWave < len) l[r] = L[min(r * kWave + lane, len - 1)];
      }
#pragma unroll
      for (uint32_t r = 0; r < kPackRegs; ++r) {
        p[r] = a.word(l[r]);
        dst[r] = 0;
      }
      uint32_t run = 0, upto = 0;  // upto: lane x, labels of hop <= x
      for (uint32_t x = 0; x <= a.K; ++x) {
#pragma unroll
        for (uint32_t r = 0; r < kPackRegs; ++r) {
          if (r * kWave >= len) break;
          const bool here = __builtin_amdgcn_ubfe(p[r], a.db, a.hsh - a.db) == x;
          unsigned long long m = __ballot(here);
          if (len - r * kWave < kWave) m &= (1ull << (len - r * kWave)) - 1ull;
          if (here)
            dst[r] = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                               __builtin_amdgcn_mbcnt_lo((uint32_t)m, run));
          run += (uint32_t)__popcll(m);
        }
        if (lane == x) upto = run;
      }
      if (lane < a.K) a.hcnt[(v0 + i) * a.K + lane] = upto;
#pragma unroll
      for (uint32_t r = 0; r < kPackRegs; ++r)
        if (r * kWave + lane < len) T[dst[r]] = p[r];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (uint32_t r = 0; r < kPackRegs; ++r)
        if (r * kWave + lane < len) a.out[b + r * kWave + lane] = T[r * kWave + lane];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
}

// Longer lists: counted, then read again and scattered, kPackStep * 64 labels in
// flight.  Lane i looks at list wave + i * waves, so that long lists, which lie
// together, spread over the waves.  (A workgroup per list that held it in registers:
// 1,150 us for the longer lists of R-MAT 262,144, this form 600.)
constexpr uint32_t kPackStep = 4;
__global__ void __launch_bounds__(kQThreads) k_pack_long(PackArgs a) {
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t wave = blockIdx.x * kQWaves + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t nwaves = gridDim.x * kQWaves;
  for (uint64_t v0 = wave; v0 < a.n; v0 += nwaves * kWave) {
    const uint64_t vi = min<uint64_t>(v0 + lane * nwaves, a.n - 1);
    for (unsigned long long todo =
             __ballot(v0 + lane * nwaves < a.n &&
                      a.off[vi + 1] - a.off[vi] > (unsigned long long)kPackHeld);
         todo; todo &= todo - 1) {
      const uint64_t v = v0 + (uint32_t)(__ffsll((long long)todo) - 1) * nwaves;
      const unsigned long long b = a.off[v];
      const uint32_t len = (uint32_t)(a.off[v + 1] - b);
      const unsigned long long *L = a.lab + b;
      // every label with its hop (past the end: no hop)
      auto each = [&](auto &&use) {
        for (uint32_t j0 = 0; j0 < len; j0 += kPackStep * kWave) {
          unsigned long long l[kPackStep];
#pragma unroll
          for (uint32_t r = 0; r < kPackStep; ++r)
            l[r] = L[min(j0 + r * kWave + lane, len - 1)];
#pragma unroll
          for (uint32_t r = 0; r < kPackStep; ++r)
            if (j0 + r * kWave < len)
              use(l[r], j0 + r * kWave + lane < len ? label_hop(l[r]) : kInf32);
        }
      };
      uint32_t pos[kMaxK + 1];
#pragma unroll
      for (uint32_t x = 0; x <= kMaxK; ++x) pos[x] = 0;
      each([&](unsigned long long, uint32_t hop) {
#pragma unroll
        for (uint32_t x = 0; x <= kMaxK; ++x)
          if (x <= a.K) pos[x] += (uint32_t)__popcll(__ballot(hop == x));
      });
      uint32_t run = 0;
#pragma unroll
      for (uint32_t x = 0; x <= kMaxK; ++x) {
        const uint32_t c = pos[x];
        pos[x] = run;
        run += c;
        if (x < a.K && lane == 0) a.hcnt[v * a.K + x] = run;
      }
      each([&](unsigned long long l, uint32_t hop) {
        uint32_t dst = 0;
#pragma unroll
        for (uint32_t x = 0; x <= kMaxK; ++x) {
          if (x > a.K) continue;
          const unsigned long long m = __ballot(hop == x);
          if (hop == x)
            dst = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m, pos[x]));
          pos[x] += (uint32_t)__popcll(m);
        }
        if (hop != kInf32) a.out[b + dst] = a.word(l);
      });
    }
  }
}

static uint32_t bits_for(uint64_t x) {  // bits that hold 0..x, at least 1
  uint32_t b = 1;
  while (b < 64 && (x >> b)) ++b;
  return b;
}

// Makes the index's 32-bit query copy on stream st when the fields fit 32
// bits (hub bits of n - 1, hop bits of K, dist bits of the index's distance
// bound), once per label set, and waits for it; tuning knob HSDL_QUERY32=0
// keeps the 8-byte labels.
static std::mutex g_q32_mu;
static int ensure_query32(const hsdl_index *idx, hipStream_t st) {
  std::lock_guard<std::mutex> g(g_q32_mu);
  if (idx->q32.load(std::memory_order_acquire)) return HSDL_OK;
  const uint32_t hb = bits_for(idx->n ? idx->n - 1u : 0u), pb = bits_for(idx->K),
                 db = bits_for(idx->dist_max);
  if (hb + pb + db > 32) {
    idx->q32.store(2, std::memory_order_release);
    return HSDL_OK;
  }
  // the copy is an optimisation: without room for it, queries read the
  // 8-byte labels.  The prefix counts lie after the labels.
  if (idx->lab32.alloc((idx->total + (uint64_t)idx->n * idx->K) * 4) != HSDL_OK) {
    idx->q32.store(2, std::memory_order_release);
    return HSDL_OK;
  }
  const uint32_t grid = (uint32_t)std::min<uint64_t>(4096, idx->n / kQWaves + 1ull);
  const PackArgs a{idx->n,
                   (uint32_t)idx->K,
                   idx->off.as<unsigned long long>(),
                   idx->lab.as<unsigned long long>(),
                   idx->lab32.as<uint32_t>(),
                   idx->lab32.as<uint32_t>() + idx->total,
                   pb + db,
                   db};
  hipLaunchKernelGGL(k_pack_short, dim3(grid), dim3(kQThreads), 0, st, a);
  hipLaunchKernelGGL(k_pack_long, dim3(grid), dim3(kQThreads), 0, st, a);
  HSDL_HIP(hipGetLastError());
  // queries on other streams may read the copy as soon as it is marked made
  HSDL_HIP(hipStreamSynchronize(st));
  idx->q32_hop_bits = pb;
  idx->q32_dist_bits = db;
  idx->q32.store(1, std::memory_order_release);
  return HSDL_OK;
}

int prepare_query(const hsdl_index *idx) {
  if (!env_u32("HSDL_QUERY32", 1, 0, 1) || idx->q32.load(std::memory_order_acquire))
    return HSDL_OK;
  return ensure_query32(idx, nullptr);
}

// Table slots per wave: a list part is a few hundred labels, hashed at a load
// of a quarter where the table has room; 1,024 slots are 16 KB per workgroup
// and keep a CU's 32 waves resident.  2^21 queries of R-MAT 2^20 vertices (1,218
// labels per list) with 512 / 1,024 / 2,048 / 4,096 slots: 5.05 / 4.70 / 8.4 / 8.7 ms;
// of 262,144 (672): 3.20 / 2.80 / 4.5 / 5.5.  Tuning knob HSDL_QUERY_SLOTS (a power of
// two from 64).
static uint32_t query_slots() { return pow2_at_most(env_u32("HSDL_QUERY_SLOTS", 1024, 64, 4096)); }

static uint64_t mean_labels(const hsdl_index *idx) { return idx->n ? idx->total / idx->n : 0; }

// Whether a call's queries get a workgroup each: up to a quarter of the square of
// the mean list length, within [2,048, 131,072].  A call ends with its longest list's
// query, and a call of few queries leaves waves idle beside it; many queries fill
// the chip anyway, and a wave per query does the less work.  Team / wave, us:
//   672 labels per list (R-MAT 262,144, K = 5): 8,192 queries 61 / 94, 65,536 211 / 230,
//   131,072 385 / 337
//   349 (65,536, K = 4): 32,768 120 / 105, 65,536 181 / 113; 8-byte labels 16,384 67 / 80
//   123 (16,384, K = 4), 8-byte: 2,048 20 / 22, 4,096 24 / 23, 16,384 48 / 37
// Calls in flight together (shared: a server's batches) have the chip filled by each
// other: there up to 32,768 at most.
// Up to 1,024 queries, or 2,048 of long lists, a team has eight waves: 672 labels,
// four / eight: 512 27 / 22, 2,048 37 / 35; 1,209: 2,048 60 / 50; 349: 2,048 25 / 27.
// Tuning knob HSDL_QUERY_TEAM: the most queries of a team call.
static bool use_team(const hsdl_index *idx, uint64_t nq, bool shared) {
  const uint64_t mean = std::min<uint64_t>(mean_labels(idx), 1024);
  const uint64_t most =
      std::min<uint64_t>(std::max<uint64_t>(mean * mean / 4, 2048), shared ? 1u << 15 : 1u << 17);
  return nq <= env_u32("HSDL_QUERY_TEAM", (uint32_t)most, 0, 0xFFFFFFFFu);
}
static bool use_wide(const hsdl_index *idx, uint64_t nq) {
  return nq <= (mean_labels(idx) > 512 ? 2048 : 1024);
}

// Whether a call reads the query copy, where there is one.  A query over it goes
// through more round trips (prefix counts, table) for fewer labels, so small calls
// and short lists read the 8-byte labels: up to 3 * 2^30 of queries times the
// square of the mean list length.  8-byte / copy, us:
//   123 labels per list: 16,384 queries 37 / 61, 131,072 119 / 132
//   349: 1,024 20 / 27, 16,384 67 / 70, 32,768 109 / 105
//   672: 1,024 27 / 30, 4,096 49 / 47, 8,192 71 / 61
//   1,209: 1,024 36 / 40, 4,096 70 / 69, 8,192 109 / 93
// (a workgroup of four waves per query over both lists, hub-ordered: 21, 24, 29
// and 45 at 1,024).  HSDL_QUERY32=1 always reads the copy.
static bool use_copy(const hsdl_index *idx, uint64_t nq) {
  if (getenv("HSDL_QUERY32")) return true;
  const double mean = (double)mean_labels(idx);
  return (double)nq * mean * mean > 3.0 * 0x1p30;
}

int launch_query(const hsdl_index *idx, size_t nq, const uint32_t *d_s, const uint32_t *d_t,
                 const int8_t *d_k, int32_t *d_out, hipStream_t st, bool may_alloc,
                 bool shared) {
  if (nq == 0) return HSDL_OK;
  const bool want32 = env_u32("HSDL_QUERY32", 1, 0, 1) != 0;
  if (want32 && may_alloc && !idx->q32.load(std::memory_order_acquire)) {
    // a stream under graph capture takes no allocation or synchronisation
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HSDL_HIP(hipStreamIsCapturing(st, &cs));
    if (cs == hipStreamCaptureStatusNone) {
      const int rc = ensure_query32(idx, st);
      if (rc) return rc;
    }
  }
  const bool copy =
      want32 && idx->q32.load(std::memory_order_acquire) == 1 && use_copy(idx, nq);
  const uint32_t slots = copy ? query_slots() : 0;
  const size_t lds = copy ? (size_t)slice_words(slots) * 4 * kQWaves : 0;
  const bool team = use_team(idx, nq, shared);
  const bool wide = team && use_wide(idx, nq) && lds <= 32 * 1024;  // 64 KB at most
  const uint32_t threads = wide ? 2 * kQThreads : kQThreads;
  const uint32_t fill = query_grid(idx->device, copy, lds) / (threads / kQThreads);
  const uint32_t grid =
      (uint32_t)std::min<uint64_t>(team ? nq : (nq + kQWaves - 1) / kQWaves, std::max(1u, fill));
  if (copy) {
    const uint32_t db = idx->q32_dist_bits, pb = idx->q32_hop_bits;
    hipLaunchKernelGGL(wide ? k_query32_team<2 * kQThreads>
                            : team ? k_query32_team<kQThreads> : k_query32,
                       dim3(grid), dim3(threads), lds * (threads / kQThreads), st,
                       Lab32{db, pb + db, (1u << pb) - 1u, (1u << db) - 1u}, idx->n,
                       (uint32_t)idx->K, idx->off.as<unsigned long long>(),
                       idx->lab32.as<uint32_t>(), idx->lab32.as<uint32_t>() + idx->total,
                       idx->hubs_below ? 1u : 0u, (uint64_t)nq, d_s, d_t, d_k, d_out,
                       team ? slots * (threads / kWave) : slots, idx->lab.as<unsigned long long>());
  } else {
    hipLaunchKernelGGL(wide ? k_query64_team<2 * kQThreads>
                            : team ? k_query64_team<kQThreads> : k_query64,
                       dim3(grid), dim3(threads), 0, st, idx->n,
                       idx->off.as<unsigned long long>(), idx->lab.as<unsigned long long>(),
                       (uint64_t)nq, d_s, d_t, d_k, d_out);
  }
  HSDL_HIP(hipGetLastError());
  return HSDL_OK;
}

}  // namespace hsdl

using namespace hsdl;

extern "C" {

int hsdl_query_device(const hsdl_index *idx, size_t n, const uint32_t *d_s, const uint32_t *d_t,
                      const int8_t *d_k, int32_t *d_out, void *hip_stream) {
  if (!idx) return fail(HSDL_EINVAL, "null index");
  if (n && (!d_s || !d_t || !d_k || !d_out)) return fail(HSDL_EINVAL, "null query buffers");
  return launch_query(idx, n, d_s, d_t, d_k, d_out, (hipStream_t)hip_stream);
}

static int query_body(const hsdl_index *idx, size_t n, const uint32_t *s, const uint32_t *t,
               const int8_t *k, int32_t *out) {
  if (!idx) return fail(HSDL_EINVAL, "null index");
  if (n == 0) return HSDL_OK;
  if (!s || !t || !k || !out) return fail(HSDL_EINVAL, "null query arrays");
  if (!all_below(s, t, n, idx->n)) return fail(HSDL_EINVAL, "query vertex out of range");
  int dev = 0;
  int rc = use_device(idx->device, &dev);
  if (rc) return rc;
  // the kernel reads the requests from pinned memory and writes the answers
  // there; a slot's copies run beside the other slot's queries
  constexpr size_t kPart = (size_t)1 << 18;
  static_assert(kPart * 13 <= kStageBytes, "a part fits a slot");
  StageLease stage;
  if ((rc = stage.take(dev, std::min(n, kPart) * 13, n > kPart ? 2 : 1))) return rc;
  const size_t part = std::min(n, kPart);
  size_t sent = 0, first[2] = {0, 0}, cnt[2] = {0, 0};
  for (int x = 0;; x ^= 1) {
    uint8_t *h = stage->h[x];
    uint32_t *hs = reinterpret_cast<uint32_t *>(h), *ht = hs + part;
    int32_t *ho = reinterpret_cast<int32_t *>(ht + part);
    int8_t *hk = reinterpret_cast<int8_t *>(ho + part);
    if (cnt[x]) {
      if ((rc = stage->wait(x))) return rc;
      std::memcpy(out + first[x], ho, cnt[x] * 4);
      cnt[x] = 0;
    }
    if (sent < n) {
      const size_t m = std::min(part, n - sent);
      std::memcpy(hs, s + sent, m * 4);
      std::memcpy(ht, t + sent, m * 4);
      std::memcpy(hk, k + sent, m);
      if ((rc = launch_query(idx, m, hs, ht, hk, ho, stage->st)) || (rc = stage->sent(x))) return rc;
      first[x] = sent;
      cnt[x] = m;
      sent += m;
    } else if (!cnt[x ^ 1]) {
      return HSDL_OK;
    }
  }
}

int hsdl_query(const hsdl_index *idx, size_t n, const uint32_t *s, const uint32_t *t,
               const int8_t *k, int32_t *out) {
  return hsdl::guarded([&] { return query_body(idx, n, s, t, k, out); });
}

}  // extern "C"

// ------------------------------------------------------- no-allocation query
// hsdl_query_noalloc stages the requests and answers in `scratch`, a
// file-scope device array that every GPU the library runs on holds until the
// process ends, instead of allocating device buffers per call: for callers
// that cannot allocate.  Layout for n <= kNoAllocMaxQueries requests:
//   [s: u32 x max][t: u32 x max][out: i32 x max][k: i8 x max]
// Nothing in it must start at zero (the query kernel writes every answer).
// Every call on one GPU shares that GPU's array: calls that overlap on one
// GPU race and must be serialised by the caller.
namespace {
constexpr size_t kNoAllocMaxQueries = (size_t)1 << 20;
constexpr size_t kNoAllocBytes = kNoAllocMaxQueries * 13;
static_assert(HSDL_NOALLOC_MAX_QUERIES == kNoAllocMaxQueries, "header and library disagree");
constexpr int kNoAllocDevices = 64;
}  // namespace

static __device__ __align__(256) uint8_t scratch[kNoAllocBytes];

namespace {
// Device address of `scratch` per device: the host-side name is only a
// stand-in, so host code uses these (looked up once per device, with that
// device current).
std::mutex g_scratch_mu;
void *g_scratch_ptr[kNoAllocDevices] = {};

int scratch_for_device(int dev, uint8_t **out) {
  if (dev < 0 || dev >= kNoAllocDevices) return fail(HSDL_ENODEV, "device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return hip_fail(e, "hipGetSymbolAddress(scratch)", __FILE__, __LINE__);
    g_scratch_ptr[dev] = p;
  }
  *out = static_cast<uint8_t *>(g_scratch_ptr[dev]);
  return HSDL_OK;
}
}  // namespace

extern "C" {

static int query_noalloc_body(const hsdl_index *idx, size_t n, const uint32_t *s,
                              const uint32_t *t, const int8_t *k, int32_t *out) {
  if (!idx) return fail(HSDL_EINVAL, "null index");
  if (n > kNoAllocMaxQueries)
    return fail(HSDL_EINVAL, "hsdl_query_noalloc takes at most HSDL_NOALLOC_MAX_QUERIES (2^20) "
                             "queries per call");
  if (n == 0) return HSDL_OK;
  if (!s || !t || !k || !out) return fail(HSDL_EINVAL, "null query arrays");
  if (!all_below(s, t, n, idx->n)) return fail(HSDL_EINVAL, "query vertex out of range");
  int dev = 0;
  int rc = use_device(idx->device, &dev);
  if (rc) return rc;
  uint8_t *base = nullptr;
  if ((rc = scratch_for_device(dev, &base))) return rc;
  uint32_t *ds = reinterpret_cast<uint32_t *>(base);
  uint32_t *dt = ds + kNoAllocMaxQueries;
  int32_t *dout = reinterpret_cast<int32_t *>(dt + kNoAllocMaxQueries);
  int8_t *dk = reinterpret_cast<int8_t *>(dout + kNoAllocMaxQueries);
  HSDL_HIP(hipMemcpy(ds, s, n * 4, hipMemcpyHostToDevice));
  HSDL_HIP(hipMemcpy(dt, t, n * 4, hipMemcpyHostToDevice));
  HSDL_HIP(hipMemcpy(dk, k, n, hipMemcpyHostToDevice));
  if ((rc = launch_query(idx, n, ds, dt, dk, dout, nullptr, false))) return rc;
  HSDL_HIP(hipMemcpy(out, dout, n * 4, hipMemcpyDeviceToHost));
  return HSDL_OK;
}

int hsdl_query_noalloc(const hsdl_index *idx, size_t n, const uint32_t *s, const uint32_t *t,
                       const int8_t *k, int32_t *out) {
  return hsdl::guarded([&] { return query_noalloc_body(idx, n, s, t, k, out); });
}

}  // extern "C"
