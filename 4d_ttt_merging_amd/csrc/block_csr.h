// What one work-group of 1,024 threads does over a list: scans, ordered ranks, and a stable CSR
// of some thousand items in LDS.
#pragma once

#include "vgo_common.h"

namespace vgo {

constexpr int kBlockThreads = 1024;
constexpr int kBlockWaves = kBlockThreads / 64;

// Exclusive prefix sum over the work-group (kBlockThreads threads); returns the
// thread's exclusive prefix and writes the total to *total.
__device__ inline int block_exclusive_scan(int v, int* lds_waves, int* total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) lds_waves[wave] = x;
  __syncthreads();
  if (wave == 0) {
    int w = lane < kBlockWaves ? lds_waves[lane] : 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(w, off);
      if (lane >= off) w += y;
    }
    if (lane < kBlockWaves) lds_waves[lane] = w;  // inclusive scan of wave totals
  }
  __syncthreads();
  const int wave_base = wave > 0 ? lds_waves[wave - 1] : 0;
  const int t = lds_waves[kBlockWaves - 1];
  __syncthreads();
  *total = t;
  return wave_base + x - v;
}

// Ranks, in index order, of the elements whose flag is set: element i = c*kBlockThreads
// + tid of chunk c.  Chunks are processed 64 at a time: per (chunk, wave) counts
// from ballots go to LDS, one block scan over those 1024 counts gives every
// (chunk, wave) its offset, and a lane adds the set flags of lower lanes.
// `flag(c)` is evaluated twice per chunk; `emit(c, rank)` is called for every
// set flag.  Returns the number of set flags.
template <typename Flag, typename Emit>
__device__ inline int ordered_ranks(int n_chunks, Flag flag, Emit emit, int* cnt_lds, int* scan_lds) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int running = 0;
  for (int c0 = 0; c0 < n_chunks; c0 += 64) {
    const int nc = min(64, n_chunks - c0);
    if (static_cast<int>(threadIdx.x) >= nc * kBlockWaves) cnt_lds[threadIdx.x] = 0;
    for (int c = 0; c < nc; ++c) {
      const uint64_t m = __ballot(flag(c0 + c));
      if (lane == 0) cnt_lds[c * kBlockWaves + wave] = __popcll(m);
    }
    __syncthreads();
    const int mine = cnt_lds[threadIdx.x];  // kBlockThreads == 64 * kBlockWaves entries
    int sum = 0;
    const int pre = block_exclusive_scan(mine, scan_lds, &sum);
    cnt_lds[threadIdx.x] = pre;
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
    for (int c = 0; c < nc; ++c) {
      const bool f = flag(c0 + c);
      const uint64_t m = __ballot(f);
      if (f) emit(c0 + c, running + cnt_lds[c * kBlockWaves + wave] + __popcll(m & below));
    }
    running += sum;
    __syncthreads();
  }
  return running;
}

// Flags of up to 64 chunks of 1,024 elements, a bit per chunk: `load(c0)` gives those of chunks
// c0 .. c0 + 7 (its loads are in flight together).
template <typename Load>
__device__ __forceinline__ uint64_t chunk_bits(int n_chunks, Load load) {
  uint64_t bits = 0;
  for (int c0 = 0; c0 < n_chunks; c0 += 8) bits |= static_cast<uint64_t>(load(c0)) << c0;
  return bits;
}

// Clusters over this many items are put in order by the whole work-group, one after another.
constexpr int kBigCluster = 128;
template <int C>
struct BlockCsrLds {
  int scan[kBlockWaves];
  int n_big;
  int big[C * kBlockThreads / kBigCluster];
  int part[2][C * kBlockWaves];
};

// Counts an item of `cluster` (< 65,536; two 16-bit counters per word) and returns its place:
// cluster | slot within it << 16, the slots in no particular order.  Called by a wave's first
// lanes.  Counters of one address take turns, so where lanes four apart (the corners of a source
// are neighbours) meet in a cluster, a wave first counts that cluster once for all its lanes:
// a CSR of 12,288 items, half of them in one cluster, takes 21 us so, 51 with a counter's turn each.
__device__ __forceinline__ uint32_t take_place(uint32_t* cnt32, int cluster) {
  const int lane = threadIdx.x & 63;
  const int shift = 16 * (cluster & 1);
  int slot = -1;
#pragma unroll
  for (int round = 0; round < 2; ++round) {
    // Lane - 4 within the row of 16 (row_shr:4); -1, no cluster, for a row's first four.
    const int other = __builtin_amdgcn_update_dpp(-1, cluster, 0x114, 0xF, 0xF, false);
    const uint64_t pairs = __ballot(slot < 0 && other == cluster);
    if (pairs == 0) break;
    const int leader = __ffsll(static_cast<long long>(pairs)) - 1;
    const uint64_t same = __ballot(cluster == __shfl(cluster, leader));
    uint32_t old = 0;
    if (lane == leader) old = atomicAdd(&cnt32[cluster >> 1], static_cast<uint32_t>(__popcll(same)) << shift);
    old = __shfl(old, leader);
    if ((same >> lane) & 1ull)
      slot = static_cast<int>((old >> shift) & 0xFFFFu) + __popcll(same & ((1ull << lane) - 1ull));
  }
  if (slot < 0) slot = static_cast<int>((atomicAdd(&cnt32[cluster >> 1], 1u << shift) >> shift) & 0xFFFFu);
  return static_cast<uint32_t>(cluster) | static_cast<uint32_t>(slot) << 16;
}

// Members of clusters 0..clusters - 1 (and of the overflow cluster `clusters`, last) in item
// order, and their offsets.  Thread t holds the places of items t, t + 1024, ... (at most C) and
// cnt[0, clusters] their counts (a __syncthreads() since the last); cnt has clusters + 2 entries
// and slot n.  size(k, n) is called once per cluster.
//
// An item's rank within its cluster is the count of smaller items among the members, so a
// cluster of n members costs n^2 comparisons; for clusters over kBigCluster (identical frames
// put thousands of tokens on one destination) the waves count their members instead, at one
// barrier per cluster.
template <int C, int M, typename Size>
__device__ __forceinline__ void block_csr(const uint32_t (&place)[C], int n, int clusters, uint16_t* slot,
                                          uint16_t* cnt, BlockCsrLds<M>& lds, uint32_t* __restrict__ order,
                                          int32_t* __restrict__ offsets, Size size) {
  static_assert(C <= M && C % 4 == 0, "one big cluster per kBigCluster items; whole counts per lane");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int chunks = (n + kBlockThreads - 1) / kBlockThreads;
  if (tid == 0) lds.n_big = 0;
  __syncthreads();
  const int per = (clusters + 1 + kBlockThreads - 1) / kBlockThreads;
  const int k0 = min(clusters + 1, tid * per), k1 = min(clusters + 1, k0 + per);
  int sum = 0;
  for (int k = k0; k < k1; ++k) {
    const int m = cnt[k];
    sum += m;
    if (m > kBigCluster) lds.big[atomicAdd(&lds.n_big, 1)] = k;
  }
  int all = 0;
  int run = block_exclusive_scan(sum, lds.scan, &all);
  for (int k = k0; k < k1; ++k) {
    const int m = cnt[k];
    cnt[k] = static_cast<uint16_t>(run);
    run += m;
  }
  if (tid == 0) cnt[clusters + 1] = static_cast<uint16_t>(n);
  __syncthreads();
  for (int k = tid; k <= clusters; k += kBlockThreads) {
    offsets[k] = cnt[k];
    if (k < clusters) size(k, cnt[k + 1] - cnt[k]);
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = c * kBlockThreads + tid;
    if (c < chunks && i < n) slot[cnt[place[c] & 0xFFFFu] + (place[c] >> 16)] = static_cast<uint16_t>(i);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = c * kBlockThreads + tid;
    if (c < chunks && i < n) {
      const int cluster = place[c] & 0xFFFFu;
      const int b = cnt[cluster], e = cnt[cluster + 1];
      if (e - b <= kBigCluster) {
        int rank = 0;
        for (int j = b; j < e; ++j) rank += slot[j] < i;
        order[b + rank] = static_cast<uint32_t>(i);
      }
    }
  }
  const uint64_t below = (1ull << lane) - 1ull;
  constexpr int kPer = C / 4;  // counts of (chunk, wave) per lane, in item order
  for (int g = 0; g < lds.n_big; ++g) {
    const int cluster = lds.big[g];
    int* part = lds.part[g & 1];
    auto mine = [&](int c) {
      const int i = c * kBlockThreads + tid;
      return c < chunks && i < n && static_cast<int>(place[c] & 0xFFFFu) == cluster;
    };
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint64_t m = __ballot(mine(c));
      if (lane == 0) part[c * kBlockWaves + wave] = __popcll(m);
    }
    __syncthreads();
    int v[kPer], before = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      v[q] = part[lane * kPer + q];
      before += v[q];
    }
    const int own = before;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(before, off);
      if (lane >= off) before += y;
    }
    before -= own;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int e = c * kBlockWaves + wave;
      int pos = cnt[cluster] + __shfl(before, e / kPer);
#pragma unroll
      for (int q = 0; q + 1 < kPer; ++q) pos += q < e % kPer ? __shfl(v[q], e / kPer) : 0;
      const bool f = mine(c);
      const uint64_t m = __ballot(f);
      if (f) order[pos + __popcll(m & below)] = static_cast<uint32_t>(c * kBlockThreads + tid);
    }
  }
}

}  // namespace vgo
