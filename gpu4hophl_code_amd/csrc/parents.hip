// parents.hip -- parent vertices of the labels and hop-constrained
// shortest-path extraction.
//
// Parents.  The reference stores, with every label (hub, h, d) of vertex y,
// the vertex before y on the hub's path (Hybrid_Generation_Clean/src/
// label_gen.cu:531-541 keeps the first frontier vertex its scan meets at the
// minimum, which depends on the scan order).  Here the parent is fixed by a
// rule: the smallest frontier vertex of round h that reaches y at distance d.
// The frontier of round h is the set of vertices holding a round-(h-1) label
// of the hub, so after generation the parent is a function of the finished
// label set and the graph:
//   hop 0:  y itself (the self label)
//   hop 1:  the hub (the round-1 frontier is the hub alone)
//   hop h:  min { x in N(y) : (hub, h-1, d - w(x,y)) in L(x) }
// k_derive_parents evaluates it on the uncleaned index (the clean may remove
// the (hub, h-1) label of x); the clean then carries the parents of the
// labels it keeps.  The generation kernels are untouched.
//
// Paths.  hop_constrained_extract_shortest_path
// (CPU_HopHL/include/HBPLL/hop_constrained_two_hop_labels.h:224-319): merge
// L(s) and L(t) like the distance query, take the first pair in merge order
// (hub, then position in L(s), then position in L(t)) at the smallest dist
// sum with hop sum <= k, emit (s, parent) and (t, parent) for the pair's
// labels where the parent is not the endpoint itself, move the endpoints,
// lower k by one per edge and repeat until s == t or no pair qualifies.
// k_paths runs it with one wavefront per query.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "device.hpp"

namespace hsdl {

// first position in [lo, hi) of the sorted keys L whose key >= key
__device__ inline unsigned long long lower_bound_key(const unsigned long long *L,
                                                     unsigned long long lo, unsigned long long hi,
                                                     unsigned long long key) {
  while (lo < hi) {
    const unsigned long long mid = (lo + hi) >> 1;
    if (L[mid] < key) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// One wavefront per vertex y; lanes take 64 labels of L(y) at a time and
// walk y's id-sorted row together until every lane has found its parent
// (the first match in row order is the smallest id).  A label whose rule
// finds no neighbour (labels not made by K-round generation) counts in
// *missing and gets the vertex itself.
__global__ void __launch_bounds__(256) k_derive_parents(uint32_t n,
                                                        const unsigned long long *__restrict__ off,
                                                        const unsigned long long *__restrict__ lab,
                                                        const unsigned long long *__restrict__ goff,
                                                        const uint2 *__restrict__ adj,
                                                        uint32_t *__restrict__ par,
                                                        unsigned long long *missing) {
  const int lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / kWave;
  unsigned long long lost = 0;
  for (uint32_t y = wave; y < n; y += nwaves) {
    const unsigned long long b = off[y], e = off[y + 1];
    const unsigned long long rb = goff[y], re = goff[y + 1];
    for (unsigned long long i0 = b; i0 < e; i0 += kWave) {
      const unsigned long long i = i0 + (unsigned long long)lane;
      const bool valid = i < e;
      const unsigned long long l = valid ? lab[i] : 0ull;
      const uint32_t hub = label_hub(l), hop = label_hop(l), d = label_dist(l);
      uint32_t p = y;
      bool need = false;
      if (valid) {
        if (hop == 1) p = hub;
        else if (hop > 1) need = true;
      }
      for (unsigned long long r = rb; r < re && __ballot(need); ++r) {
        const uint2 ed = adj[r];
        if (need && ed.y <= d) {
          const unsigned long long key = pack_label(hub, hop - 1, d - ed.y);
          const unsigned long long xe = off[ed.x + 1];
          const unsigned long long pos = lower_bound_key(lab, off[ed.x], xe, key);
          if (pos < xe && lab[pos] == key) {
            p = ed.x;
            need = false;
          }
        }
      }
      if (need) ++lost;
      if (valid) par[i] = p;
    }
  }
  lost = wave_sum_u64(lost);
  if (lane == 0 && lost) atomicAdd(missing, lost);
}

// Wave-wide lexicographic minimum of (k1, k2); every lane gets the winner.
__device__ inline void wave_argmin2(unsigned long long &k1, unsigned long long &k2) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long o1 = __shfl_xor(k1, o, kWave);
    const unsigned long long o2 = __shfl_xor(k2, o, kWave);
    if (o1 < k1 || (o1 == k1 && o2 < k2)) {
      k1 = o1;
      k2 = o2;
    }
  }
}

// One wavefront per query.  Each step: lanes take labels of the shorter list,
// find the hub's run in a piece of the longer one staged in LDS by binary
// search and scan it in hop order (stopping at the first hop sum above k, like
// the reference's inner loop); the wave then takes the minimum of (dist sum,
// hub, position in L(s), position in L(t)), the pair the reference's merge
// meets first at the minimum.  A step is a chain of searches: with every probe
// a load from L2, 2^17 queries on R-MAT 65,536, K = 5, took 0.88 ms, with the
// searched list in LDS 0.45 ms (host arrays and copies included 1.49 -> 0.84).
constexpr uint32_t kPathPiece = 512;  // labels, 4 KB per wave
// A list of more than kPathSearchLen labels and kPathSearchRatio times the other is
// searched in memory: 50,000 paths between lists of 9 and 60,000 labels 1.32 -> 0.27
// ms with their copies, of 5 and 4,000 0.29 -> 0.25.
constexpr uint32_t kPathSearchLen = 2048;
constexpr uint32_t kPathSearchRatio = 64;
__global__ void __launch_bounds__(256) k_paths(size_t nq, const unsigned long long *__restrict__ off,
                                               const unsigned long long *__restrict__ lab,
                                               const uint32_t *__restrict__ par,
                                               const uint32_t *__restrict__ qs,
                                               const uint32_t *__restrict__ qt,
                                               const int8_t *__restrict__ qk, uint32_t cap,
                                               uint32_t *__restrict__ edges,
                                               uint32_t *__restrict__ counts) {
  __shared__ unsigned long long stage[256 / kWave][kPathPiece];
  const int lane = lane_id();
  const uint32_t wib = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  lds_ptr<unsigned long long> P = (lds_ptr<unsigned long long>)stage[wib];
  const size_t wave = blockIdx.x * (size_t)(256 / kWave) + wib;
  const size_t nwaves = gridDim.x * (size_t)(256 / kWave);
  for (size_t q = wave; q < nq; q += nwaves) {
    uint32_t s = __builtin_amdgcn_readfirstlane(qs[q]), t = __builtin_amdgcn_readfirstlane(qt[q]);
    int32_t k = qk[q];
    uint32_t cnt = 0;
    uint32_t *out = edges + 2 * (size_t)cap * q;
    // the row's first 64 words are a lane's each and stored together: `edges` is host
    // memory, where a store is a packet
    uint32_t row = 0;
    auto emit = [&](uint32_t v, uint32_t parent) {
      const uint32_t at = 2 * cnt;
      if (cnt < cap) {
        if ((uint32_t)lane == at) row = v;
        if ((uint32_t)lane == at + 1) row = parent;
        if (at >= kWave && lane == 0) {
          out[at] = v;
          out[at + 1] = parent;
        }
      }
      ++cnt;
    };
    // every step that emits lowers k; a step that cannot emit ends the walk
    for (int32_t step = 0; step <= 256 && s != t; ++step) {
      const unsigned long long sb = off[s], tb = off[t];
      const uint32_t slen = (uint32_t)(off[s + 1] - sb), tlen = (uint32_t)(off[t + 1] - tb);
      unsigned long long k1 = ~0ull, k2 = ~0ull;
      // pieces of the longer list B in LDS, searched by the shorter list A's
      // labels; both are hub-sorted, so a chunk of A below a piece is never
      // read again
      const bool a_is_s = slen <= tlen;
      const unsigned long long *A = lab + (a_is_s ? sb : tb), *B = lab + (a_is_s ? tb : sb);
      const uint32_t alen = a_is_s ? slen : tlen, blen = a_is_s ? tlen : slen;
      uint32_t j0 = 0;
      // the pairs of A's label `ja` and those from position x of B[p0, p0 + m), held
      // in P, of its hub
      auto pairs = [&](auto P, uint32_t p0, uint32_t m, uint32_t x, uint32_t ja,
                       unsigned long long la) {
        const uint32_t w = label_hub(la), h1 = label_hop(la);
        for (; x < m; ++x) {
          const unsigned long long lb = P[x];
          if (label_hub(lb) != w || (int32_t)(h1 + label_hop(lb)) > k) break;
          const unsigned long long c1 =
              ((unsigned long long)(label_dist(la) + label_dist(lb)) << 32) | w;
          const uint32_t jb = p0 + x;
          const unsigned long long c2 =
              ((unsigned long long)(a_is_s ? ja : jb) << 32) | (a_is_s ? jb : ja);
          if (c1 < k1 || (c1 == k1 && c2 < k2)) {
            k1 = c1;
            k2 = c2;
          }
        }
      };
      if (blen > kPathSearchLen && (uint64_t)alen * kPathSearchRatio <= blen) {
        for (; j0 < alen; j0 += kWave) {
          const uint32_t ja = min(j0 + (uint32_t)lane, alen - 1);
          const unsigned long long la = A[ja];
          const uint32_t w = label_hub(la);
          if ((int32_t)label_hop(la) > k) continue;
          uint32_t lo = 0, hi = blen;
          while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (label_hub(B[mid]) < w) lo = mid + 1; else hi = mid;
          }
          pairs(B, 0, blen, lo, ja, la);
        }
      }
      for (uint32_t p0 = 0; p0 < blen && j0 < alen; p0 += kPathPiece) {
        const uint32_t m = min(kPathPiece, blen - p0);
        for (uint32_t i = lane; i < m; i += 4 * kWave) {
          unsigned long long l[4];
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u) l[u] = B[p0 + min(i + u * kWave, m - 1)];
#pragma unroll
          for (uint32_t u = 0; u < 4; ++u)
            if (i + u * kWave < m) P[i + u * kWave] = l[u];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint32_t lo_hub = label_hub(P[0]), hi_hub = label_hub(P[m - 1]);
        for (uint32_t j = j0; j < alen; j += kWave) {
          const uint32_t ja = min(j + (uint32_t)lane, alen - 1);
          const unsigned long long la = A[ja];
          const uint32_t w = label_hub(la), h1 = label_hop(la);
          if (__builtin_amdgcn_readlane(w, 0) > hi_hub) break;
          if (__builtin_amdgcn_readlane(w, kWave - 1) < lo_hub) {
            j0 = j + kWave;
            continue;
          }
          if (w < lo_hub || w > hi_hub || (int32_t)h1 > k) continue;
          uint32_t lo = 0, hi = m - 1;
          while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (label_hub(P[mid]) < w) lo = mid + 1; else hi = mid;
          }
          pairs(P, p0, m, lo, ja, la);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
      wave_argmin2(k1, k2);
      if (k1 == ~0ull) break;  // nothing connects within k hops
      const uint32_t p1 = __builtin_amdgcn_readfirstlane(par[sb + (k2 >> 32)]);
      const uint32_t p2 = __builtin_amdgcn_readfirstlane(par[tb + (k2 & 0xFFFFFFFFull)]);
      if (p1 == s && p2 == t) break;
      if (p1 != s) {
        emit(s, p1);
        s = p1;
        --k;
      }
      if (p2 != t) {
        emit(t, p2);
        t = p2;
        --k;
      }
    }
    // slots past the path's end read 0
    if ((uint32_t)lane < 2 * cap) out[lane] = row;
    for (uint32_t e = max(2 * min(cnt, cap), (uint32_t)kWave) + lane; e < 2 * cap; e += kWave)
      out[e] = 0;
    if (lane == 0) counts[q] = cnt;
  }
}

// Derives idx->par from the graph (device copy) and the uncleaned sorted
// labels; called by the generation before it returns the index.
int derive_parents(hsdl_index *idx, const hsdl_graph *g, hipStream_t st) {
  if (!g->d_off || !g->d_adj || g->n != idx->n)
    return fail(HSDL_EINVAL, "parents need the index's graph resident on its device");
  int rc = idx->par.alloc(std::max<uint64_t>(idx->total, 1) * 4);
  if (rc) return rc;
  DevBuf missing;
  if ((rc = missing.alloc(8))) return rc;
  HSDL_HIP(hipMemsetAsync(missing.p, 0, 8, st));
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, idx->device);
  hipLaunchKernelGGL(k_derive_parents, dim3(cus * 8), dim3(256), 0, st, idx->n,
                     idx->off.as<unsigned long long>(), idx->lab.as<unsigned long long>(),
                     static_cast<const unsigned long long *>(g->d_off),
                     static_cast<const uint2 *>(g->d_adj), idx->par.as<uint32_t>(),
                     missing.as<unsigned long long>());
  HSDL_HIP(hipGetLastError());
  unsigned long long lost = 0;
  HSDL_HIP(hipMemcpyAsync(&lost, missing.p, 8, hipMemcpyDeviceToHost, st));
  HSDL_HIP(hipStreamSynchronize(st));
  if (lost) {
    idx->par.release();
    return fail(HSDL_EDEVICE, "parent derivation found labels no neighbour explains");
  }
  idx->has_parents = true;
  return HSDL_OK;
}

}  // namespace hsdl

using namespace hsdl;

extern "C" {

static int export_parents_body(const hsdl_index *idx, uint32_t *parent) {
  if (!idx || !parent) return fail(HSDL_EINVAL, "null argument");
  if (!idx->has_parents) return fail(HSDL_EINVAL, "index has no parents (build with opts.parents = 1)");
  int rc = use_device(idx->device, nullptr);
  if (rc) return rc;
  if (idx->total)
    HSDL_HIP(hipMemcpy(parent, idx->par.p, idx->total * 4, hipMemcpyDeviceToHost));
  return HSDL_OK;
}

int hsdl_export_parents(const hsdl_index *idx, uint32_t *parent) {
  return hsdl::guarded([&] { return export_parents_body(idx, parent); });
}

static int index_set_parents_body(hsdl_index *idx, const uint32_t *parent) {
  if (!idx || (!parent && idx->total)) return fail(HSDL_EINVAL, "null argument");
  for (uint64_t i = 0; i < idx->total; ++i)
    if (parent[i] >= idx->n) return fail(HSDL_EINVAL, "parent id out of range");
  int rc = use_device(idx->device, nullptr);
  if (rc) return rc;
  DevBuf p;
  if ((rc = p.alloc(std::max<uint64_t>(idx->total, 1) * 4))) return rc;
  if (idx->total) HSDL_HIP(hipMemcpy(p.p, parent, idx->total * 4, hipMemcpyHostToDevice));
  idx->par = std::move(p);
  idx->has_parents = true;
  return HSDL_OK;
}

int hsdl_index_set_parents(hsdl_index *idx, const uint32_t *parent) {
  return hsdl::guarded([&] { return index_set_parents_body(idx, parent); });
}

static int extract_paths_body(const hsdl_index *idx, size_t n, const uint32_t *s, const uint32_t *t,
                       const int8_t *k, uint32_t cap, uint32_t *edges, uint32_t *counts) {
  if (!idx) return fail(HSDL_EINVAL, "null index");
  if (n == 0) return HSDL_OK;
  if (!s || !t || !k || !counts || (cap && !edges)) return fail(HSDL_EINVAL, "null path arrays");
  if (!idx->has_parents) return fail(HSDL_EINVAL, "index has no parents (build with opts.parents = 1)");
  if (!all_below(s, t, n, idx->n)) return fail(HSDL_EINVAL, "query vertex out of range");
  int dev = 0;
  int rc = use_device(idx->device, &dev);
  if (rc) return rc;
  // a slot: requests (9 B a query), counts and edges, read and written in place; the
  // host's part of a slot runs beside the other slot's kernel
  const size_t per = 13 + (size_t)8 * cap;
  // (a query whose edges exceed a kept slot gets slots of its own)
  const size_t most = std::max<size_t>(1, (kStageBytes - 64) / per);
  const size_t part = std::min(n, most >= 4 ? most & ~(size_t)3 : most);
  StageLease stage;
  if ((rc = stage.take(dev, part * per + 64, n > part ? 2 : 1))) return rc;
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, idx->device);
  size_t sent = 0, first[2] = {0, 0}, cnt[2] = {0, 0};
  for (int x = 0;; x ^= 1) {
    uint8_t *h = stage->h[x];
    uint32_t *hs = reinterpret_cast<uint32_t *>(h), *ht = hs + part;
    int8_t *hk = reinterpret_cast<int8_t *>(ht + part);
    uint32_t *hc = reinterpret_cast<uint32_t *>(h + ((part * 9 + 15) & ~(size_t)15));
    if (cnt[x]) {
      if ((rc = stage->wait(x))) return rc;
      std::memcpy(counts + first[x], hc, cnt[x] * 4);
      if (cap)
        std::memcpy(edges + (size_t)2 * cap * first[x], hc + part, (size_t)8 * cap * cnt[x]);
      cnt[x] = 0;
    }
    if (sent < n) {
      const size_t m = std::min(part, n - sent);
      std::memcpy(hs, s + sent, m * 4);
      std::memcpy(ht, t + sent, m * 4);
      std::memcpy(hk, k + sent, m);
      const size_t blocks = std::min<size_t>((m + 3) / 4, (size_t)cus * 16);
      hipLaunchKernelGGL(k_paths, dim3((uint32_t)blocks), dim3(256), 0, stage->st, m,
                         idx->off.as<unsigned long long>(), idx->lab.as<unsigned long long>(),
                         idx->par.as<uint32_t>(), hs, ht, hk, cap, hc + part, hc);
      HSDL_HIP(hipGetLastError());
      if ((rc = stage->sent(x))) return rc;
      fault_in(edges + (size_t)2 * cap * sent, (size_t)8 * cap * m);
      first[x] = sent;
      cnt[x] = m;
      sent += m;
    } else if (!cnt[x ^ 1]) {
      return HSDL_OK;
    }
  }
}

int hsdl_extract_paths(const hsdl_index *idx, size_t n, const uint32_t *s, const uint32_t *t,
                       const int8_t *k, uint32_t cap, uint32_t *edges, uint32_t *counts) {
  return hsdl::guarded([&] { return extract_paths_body(idx, n, s, t, k, cap, edges, counts); });
}

}  // extern "C"
