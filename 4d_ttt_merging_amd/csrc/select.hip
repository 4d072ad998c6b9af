// Rank-and-select that turns FastVGGT match scores into a merge plan.
//
// Work of vggt_omega/models/token_merging.py:1112-1121:
//   ranked  = best.argsort(descending=True, stable=True)
//   removed = sources[ranked[:r]];  target = destinations[targets[ranked[:r]]]
//   keep    = ascending non-removed ids;  inverse: kept -> compact id,
//             removed -> compact id of its target.
// Only the *set* of the r best sources matters (keep is re-sorted, inverse is
// per token), so instead of a full sort one work-group per batch element runs
// a four-pass radix select on the order-preserving 32-bit image of `best`
// (coalesced histogram passes, parallel digit search), then breaks ties at the
// threshold by source position (the stable sort's rule) and builds keep /
// inverse, both with ballot-based ordered ranks (one block scan per 64 chunks
// of 1024 elements).  Integer work, bit-exact, deterministic.
#include "block_csr.h"

namespace vgo {
namespace {

constexpr int kThreads = kBlockThreads;
constexpr int kWavesS = kBlockWaves;

// Order-preserving map float -> uint32 (NaN above +inf, -0 folded onto +0),
// matching the comparison order of torch's descending stable sort.
__device__ __forceinline__ uint32_t ord32(float x) {
  if (x != x) return 0xFFFFFFFFu;
  uint32_t b = __float_as_uint(x);
  if (b == 0x80000000u) b = 0;
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// hist[digit] += 1 for every lane with `valid`.  Keys here cluster in a few
// digits (bf16-rounded scores), and same-address LDS atomics serialise, so a
// wave first adds whole groups of equal digits through a leader lane; after a
// few groups the remaining lanes fall back to one atomic each.
__device__ __forceinline__ void hist_add(int* hist, bool valid, uint32_t digit) {
  const int lane = threadIdx.x & 63;
  uint64_t active = __ballot(valid);
#pragma unroll
  for (int round = 0; round < 4; ++round) {
    if (active == 0) return;
    const int leader = __ffsll(static_cast<long long>(active)) - 1;
    const uint32_t d = __shfl(digit, leader);
    const uint64_t same = __ballot(valid && digit == d) & active;
    if (lane == leader) atomicAdd(&hist[d], __popcll(same));
    active &= ~same;
  }
  if ((active >> lane) & 1ull) atomicAdd(&hist[digit], 1);
}

// Keys per thread held in registers (sources beyond kThreads * kKeyRegs are
// re-read from global memory in batches of the same size).
constexpr int kKeyRegs = 32;

__global__ __launch_bounds__(kThreads) void fastvggt_assemble_kernel(
    const float* __restrict__ best, const int32_t* __restrict__ target,
    const int64_t* __restrict__ source_ids, const int64_t* __restrict__ dest_ids, int ns, int nd,
    int total, int removed, int64_t* __restrict__ keep, int64_t* __restrict__ inverse,
    uint8_t* __restrict__ removed_flag) {
  __shared__ int hist[256];
  __shared__ int scan_lds[kWavesS];
  __shared__ int cnt_lds[kThreads];
  __shared__ uint32_t sel_prefix;
  __shared__ int sel_above;

  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const float* bb = best + static_cast<int64_t>(b) * ns;
  const int32_t* tb = target + static_cast<int64_t>(b) * ns;
  int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  int64_t* kp = keep + static_cast<int64_t>(b) * (total - removed);
  uint8_t* flag = removed_flag + static_cast<int64_t>(b) * ns;
  const int s_chunks = (ns + kThreads - 1) / kThreads;
  const int t_chunks = (total + kThreads - 1) / kThreads;

  // Keys of chunks [0, kKeyRegs) in registers; key(c) reads further chunks from global.
  uint32_t kreg[kKeyRegs];
#pragma unroll
  for (int c = 0; c < kKeyRegs; ++c) {
    const int i = c * kThreads + tid;
    kreg[c] = i < ns ? ord32(bb[i]) : 0u;
  }
  auto key = [&](int c) -> uint32_t {  // chunks >= kKeyRegs
    const int i = c * kThreads + tid;
    return i < ns ? ord32(bb[i]) : 0u;
  };

  // ---- radix select (8-bit digits, most significant first) of the r-th largest key.
  if (tid == 0) {
    sel_prefix = 0;
    sel_above = 0;
  }
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    const uint32_t prefix = sel_prefix;
    const uint32_t pmask = pass == 0 ? 0u : (0xFFFFFFFFu << (32 - 8 * pass));
#pragma unroll
    for (int c = 0; c < kKeyRegs; ++c) {
      if (c < s_chunks)  // wave-uniform
        hist_add(hist, c * kThreads + tid < ns && (kreg[c] & pmask) == prefix, (kreg[c] >> shift) & 0xFF);
    }
    for (int c = kKeyRegs; c < s_chunks; ++c) {
      const int i = c * kThreads + tid;
      const uint32_t o = i < ns ? ord32(bb[i]) : 0u;
      hist_add(hist, i < ns && (o & pmask) == prefix, (o >> shift) & 0xFF);
    }
    __syncthreads();
    if (tid < 64) {
      // Lane l owns digits 4l..4l+3; c(d) = keys with digit >= d.  The digit
      // sought is the largest d with c(d) >= need.
      const int need = removed - sel_above;
      int h[4], local = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        h[q] = hist[4 * lane + q];
        local += h[q];
      }
      int suffix = local;  // inclusive suffix sum over lanes >= lane
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_down(suffix, off);
        if (lane + off < 64) suffix += y;
      }
      int c = suffix - local;  // keys in digits above this lane's range
      int found = -1, above = 0;
#pragma unroll
      for (int q = 3; q >= 0; --q) {
        if (found < 0 && c + h[q] >= need) {
          found = 4 * lane + q;
          above = c;
        }
        c += h[q];
      }
      const uint64_t hit = __ballot(found >= 0);
      const int top = 63 - __clzll(hit);  // highest lane holding the digit
      if (lane == top) {
        sel_above += above;
        sel_prefix = prefix | (static_cast<uint32_t>(found) << shift);
      }
    }
    __syncthreads();
  }
  const uint32_t thresh = sel_prefix;
  const int need_ties = removed - sel_above;  // ties at the threshold to remove, lowest position first

  // ---- removed sources: keys above the threshold, and the first need_ties ties.
  // inv[t] holds 0 for kept tokens and -1 for removed ones until compaction.
  for (int t0 = 0; t0 < total; t0 += kThreads * 8) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int t = t0 + q * kThreads + tid;
      if (t < total) inv[t] = 0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < kKeyRegs; ++c) {
    const int i = c * kThreads + tid;
    if (i < ns) flag[i] = kreg[c] > thresh ? 1 : 0;
  }
#pragma unroll
  for (int c = 0; c < kKeyRegs; ++c) {
    const int i = c * kThreads + tid;
    const int64_t sid = (i < ns && kreg[c] > thresh) ? source_ids[i] : -1;
    if (sid >= 0 && sid < total) inv[sid] = -1;
  }
  for (int c = kKeyRegs; c < s_chunks; ++c) {
    const int i = c * kThreads + tid;
    if (i < ns) {
      const bool rm = key(c) > thresh;
      flag[i] = rm ? 1 : 0;
      if (rm) {
        const int64_t sid = source_ids[i];
        if (sid >= 0 && sid < total) inv[sid] = -1;
      }
    }
  }
  __syncthreads();
  uint32_t tie_bits = 0;  // chunks < kKeyRegs
#pragma unroll
  for (int c = 0; c < kKeyRegs; ++c)
    tie_bits |= (c * kThreads + tid < ns && kreg[c] == thresh ? 1u : 0u) << c;
  ordered_ranks(
      s_chunks,
      [&](int c) {
        if (c < kKeyRegs) return ((tie_bits >> c) & 1u) != 0u;
        return c * kThreads + tid < ns && key(c) == thresh;
      },
      [&](int c, int rank) {
        if (rank < need_ties) {
          const int i = c * kThreads + tid;
          flag[i] = 1;
          const int64_t sid = source_ids[i];
          if (sid >= 0 && sid < total) inv[sid] = -1;
        }
      },
      cnt_lds, scan_lds);

  // ---- compact ids of kept tokens (ascending), keep list.  Kept flags of the
  // first 64 token chunks are read once into a bit mask.
  uint64_t kept_bits = 0;
  {
    const int nc = min(t_chunks, 64);
    for (int c0 = 0; c0 < nc; c0 += 8) {
      int64_t v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int t = (c0 + q) * kThreads + tid;
        v[q] = (c0 + q < nc && t < total) ? inv[t] : -1;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) kept_bits |= (v[q] == 0 ? 1ull : 0ull) << (c0 + q);
    }
  }
  const int n_keep = total - removed;
  ordered_ranks(
      t_chunks,
      [&](int c) {
        if (c < 64) return ((kept_bits >> c) & 1ull) != 0ull;
        const int t = c * kThreads + tid;
        return t < total && inv[t] == 0;
      },
      [&](int c, int rank) {
        const int t = c * kThreads + tid;
        inv[t] = rank;
        if (rank < n_keep) kp[rank] = t;  // always true for a valid (disjoint) source list
      },
      cnt_lds, scan_lds);

  // ---- removed sources point at their target's compact id (eight independent
  // load chains per thread in flight).
  for (int c0 = 0; c0 < s_chunks; c0 += 8) {
    int64_t sid[8], dst[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int i = (c0 + q) * kThreads + tid;
      sid[q] = -1;
      dst[q] = -1;
      if (i < ns && flag[i]) {
        sid[q] = source_ids[i];
        const int32_t d = tb[i];
        dst[q] = (d >= 0 && d < nd) ? dest_ids[d] : -1;
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (sid[q] >= 0 && sid[q] < total) inv[sid[q]] = (dst[q] >= 0 && dst[q] < total) ? inv[dst[q]] : -1;
    }
  }
}


// Sparse-convex plan assembly (vggt_omega/models/sparse_convex.py:2435-2455):
//   selected = fit >= threshold; sources = candidates[selected] (ascending);
//   keep = ascending non-sources; o2c = compact id or -1;
//   parent_compact = o2c[support[selected]]; weights = alpha[selected].
// Buffers are sized for the worst case (n sources, total kept); stats[0] = M
// (sources), stats[1] = hard candidates, stats[2] = fallback candidates (copied
// from the device counter), stats[3] = sum of the selected fits.
//
// Two launches.  The first, one work-group, does what needs ranks over all
// candidates and tokens: o2c, the statistics, and the candidate of every source
// (left in the first word of its `parent` row).  Its time is the latency of its
// loads: they are coalesced and eight chunks of 1,024 are in flight.  The second
// writes the rest from the whole chip (56 bytes per source, 8 per kept token, which
// one work-group would store at a few tens of GB/s).  5,672 candidates of 8,658 tokens:
// 51 us from one work-group whose threads took contiguous runs, now 13.5 + 5.
__global__ __launch_bounds__(kThreads) void sparse_convex_select_kernel(
    const float* __restrict__ fit, const int64_t* __restrict__ candidate, const float* __restrict__ top1,
    float easy_threshold, const int* __restrict__ failed_count, int n, int total, float threshold, int64_t* o2c,
    int64_t* __restrict__ parent, float* __restrict__ stats) {
  __shared__ int scan_lds[kWavesS];
  __shared__ int cnt_lds[kThreads];
  __shared__ float red[kWavesS];
  const int tid = threadIdx.x;
  for (int t = tid; t < total; t += kThreads) o2c[t] = 0;
  __syncthreads();

  // ---- candidates, 64 chunks at a time
  int hard = 0, n_sel = 0;
  float fsum = 0.0f;
  for (int g0 = 0; g0 < n; g0 += 64 * kThreads) {
    const int chunks = min(64, (n - g0 + kThreads - 1) / kThreads);
    const uint64_t selected = chunk_bits(chunks, [&](int c0) {
      float f[8], e[8];
      int64_t id[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int r = g0 + (c0 + q) * kThreads + tid;
        f[q] = r < n ? fit[r] : 0.0f;
        e[q] = r < n && top1 ? top1[r] : 0.0f;
        id[q] = r < n ? candidate[r] : -1;
      }
      uint32_t bits = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int r = g0 + (c0 + q) * kThreads + tid;
        if (r >= n) continue;
        hard += !(top1 && e[q] >= easy_threshold);
        if (!(f[q] >= threshold)) continue;
        bits |= 1u << q;
        fsum += f[q];
        if (id[q] >= 0 && id[q] < total) o2c[id[q]] = -1;
      }
      return bits;
    });
    const int before = n_sel;
    n_sel += ordered_ranks(
        chunks, [&](int c) { return ((selected >> c) & 1ull) != 0ull; },
        [&](int c, int rank) { parent[4 * static_cast<int64_t>(before + rank)] = g0 + c * kThreads + tid; }, cnt_lds,
        scan_lds);
  }
  int n_hard = 0;
  block_exclusive_scan(hard, scan_lds, &n_hard);

  // ---- tokens
  int kept = 0;
  __syncthreads();
  for (int g0 = 0; g0 < total; g0 += 64 * kThreads) {
    const int chunks = min(64, (total - g0 + kThreads - 1) / kThreads);
    const uint64_t stays = chunk_bits(chunks, [&](int c0) {
      int64_t v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int t = g0 + (c0 + q) * kThreads + tid;
        v[q] = t < total ? o2c[t] : -1;
      }
      uint32_t bits = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) bits |= static_cast<uint32_t>(v[q] == 0) << q;
      return bits;
    });
    const int before = kept;
    kept += ordered_ranks(
        chunks, [&](int c) { return ((stays >> c) & 1ull) != 0ull; },
        [&](int c, int rank) { o2c[g0 + c * kThreads + tid] = before + rank; }, cnt_lds, scan_lds);
  }

  // Deterministic fit sum (fixed thread/wave order).
  float v = fsum;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  if (tid == 0) {
    float s = 0.0f;
    for (int w = 0; w < kWavesS; ++w) s += red[w];
    stats[0] = static_cast<float>(n_sel);
    stats[1] = static_cast<float>(n_hard);
    stats[2] = failed_count ? static_cast<float>(*failed_count) : 0.0f;
    stats[3] = s;
  }
}

__global__ __launch_bounds__(256) void sparse_convex_fill_kernel(
    const float* __restrict__ alpha, const int64_t* __restrict__ support, const int64_t* __restrict__ candidate,
    const int64_t* __restrict__ o2c, const float* __restrict__ stats, int n, int total, int64_t* __restrict__ keep,
    int64_t* __restrict__ source, int64_t* parent, float* __restrict__ weight) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < total) {
    const int64_t k = o2c[i];
    if (k >= 0) keep[k] = i;
  }
  // Four lanes per source; all four have its candidate before any stores its parent.
  const bool live = i < 4 * static_cast<int64_t>(min(n, static_cast<int>(stats[0])));
  const int r = __shfl(live && (i & 3) == 0 ? static_cast<int>(parent[i]) : -1, threadIdx.x & 60);
  if (!live || r < 0 || r >= n) return;
  const int64_t sup = support[4 * static_cast<int64_t>(r) + (i & 3)];
  weight[i] = alpha[4 * static_cast<int64_t>(r) + (i & 3)];
  parent[i] = sup >= 0 && sup < total ? o2c[sup] : -1;
  if ((i & 3) == 0) source[i >> 2] = candidate[r];
}

// ---------------------------------------------------------------------------
// Multi-work-group FastVGGT assembly (the workspace entry).  The same rule as
// fastvggt_assemble_kernel, spread over the chip as a chain of short kernels:
//   init     inverse = 0, workspace histograms cleared
//   hist p   (p = 0..3) histogram of digit p of the keys matching the prefix
//            chosen from digits 0..p-1 (each work-group re-derives that
//            prefix from the previous histogram; work-group 0 records it)
//   mark     threshold; keys above it are removed; ties counted per group
//   ties     the first need_ties ties in source order are removed
//   kcount   kept tokens per 512-token group
//   compact  compact ids (ascending) and the keep list
//   inverse  removed sources take their target's compact id
// Every step is integer work; the result is bit-identical to the one-group
// kernel.
constexpr int kAThreads = 256;
// Two elements per thread: 512-element groups spread each step over 4x the
// work-groups of 2048-element ones (47 / 65 at C4 instead of 12 / 17), which took
// the C4 plan build from 500 to 480 us.
constexpr int kAPer = 2;                     // elements per thread, contiguous
constexpr int kAChunk = kAThreads * kAPer;  // elements per work-group
constexpr int kASel = 4 * 256;               // sel[5][4] follows hist[4][256]
constexpr int kAGroupsAt = kASel + 20;       // per-group counts follow

__host__ __device__ inline int64_t fv_ws_ints(int s_groups, int t_groups) {
  return kAGroupsAt + s_groups + t_groups;
}

// Exclusive prefix over the 256 threads; *total receives the sum.
__device__ int scan256(int v, int* lds4, int* total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) lds4[wave] = x;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wave; ++w) base += lds4[w];
  const int t = lds4[0] + lds4[1] + lds4[2] + lds4[3];
  __syncthreads();
  *total = t;
  return base + x - v;
}

// Wave 0: from a 256-bin digit histogram of the keys matching `prefix`, with
// `above` keys known to lie above them, the digit of the `removed`-th largest
// key; writes the extended prefix and count above it to *out_prefix/*out_above.
__device__ void fv_select(const int* hist, uint32_t prefix, int above, int removed, int shift,
                          uint32_t* out_prefix, int* out_above) {
  const int lane = threadIdx.x & 63;
  const int need = removed - above;
  int h[4], local = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    h[q] = hist[4 * lane + q];
    local += h[q];
  }
  int suffix = local;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_down(suffix, off);
    if (lane + off < 64) suffix += y;
  }
  int c = suffix - local;
  int found = -1, more = 0;
#pragma unroll
  for (int q = 3; q >= 0; --q) {
    if (found < 0 && c + h[q] >= need) {
      found = 4 * lane + q;
      more = c;
    }
    c += h[q];
  }
  const uint64_t hit = __ballot(found >= 0);
  const int top = 63 - __clzll(hit);
  if (lane == top) {
    *out_above = above + more;
    *out_prefix = prefix | (static_cast<uint32_t>(found) << shift);
  }
}

__global__ __launch_bounds__(kAThreads) void fva_init_kernel(int total, int64_t* __restrict__ inverse,
                                                            int* __restrict__ ws, int64_t ws_ints) {
  const int b = blockIdx.y;
  int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  const int t0 = blockIdx.x * kAChunk + threadIdx.x * kAPer;
#pragma unroll
  for (int k = 0; k < kAPer; ++k)
    if (t0 + k < total) inv[t0 + k] = 0;
  if (blockIdx.x == 0) {
    int* w = ws + b * ws_ints;
    for (int i = threadIdx.x; i < kAGroupsAt; i += kAThreads) w[i] = 0;
  }
}

__global__ __launch_bounds__(kAThreads) void fva_hist_kernel(const float* __restrict__ best, int ns,
                                                            int removed, int pass, int* __restrict__ ws,
                                                            int64_t ws_ints) {
  __shared__ int lh[256];
  __shared__ uint32_t s_prefix;
  __shared__ int s_above;
  const int b = blockIdx.y;
  int* w = ws + b * ws_ints;
  const int tid = threadIdx.x;
  if (pass == 0) {
    if (tid == 0) {
      s_prefix = 0;
      s_above = 0;
    }
  } else if (tid < 64) {
    fv_select(w + (pass - 1) * 256, static_cast<uint32_t>(w[kASel + 4 * (pass - 1)]),
              w[kASel + 4 * (pass - 1) + 1], removed, 32 - 8 * pass, &s_prefix, &s_above);
  }
  lh[tid] = 0;
  __syncthreads();
  if (blockIdx.x == 0 && tid == 0) {
    w[kASel + 4 * pass] = static_cast<int>(s_prefix);
    w[kASel + 4 * pass + 1] = s_above;
  }
  const uint32_t prefix = s_prefix;
  const uint32_t pmask = pass == 0 ? 0u : (0xFFFFFFFFu << (32 - 8 * pass));
  const int shift = 24 - 8 * pass;
  const float* bb = best + static_cast<int64_t>(b) * ns;
  const int i0 = blockIdx.x * kAChunk + tid * kAPer;
#pragma unroll
  for (int k = 0; k < kAPer; ++k) {
    const int i = i0 + k;
    const uint32_t key = i < ns ? ord32(bb[i]) : 0u;
    hist_add(lh, i < ns && (key & pmask) == prefix, (key >> shift) & 0xFF);
  }
  __syncthreads();
  if (lh[tid]) atomicAdd(&w[pass * 256 + tid], lh[tid]);
}

__global__ __launch_bounds__(kAThreads) void fva_mark_kernel(const float* __restrict__ best,
                                                            const int64_t* __restrict__ source_ids,
                                                            int ns, int total, int removed,
                                                            int64_t* __restrict__ inverse,
                                                            uint8_t* __restrict__ removed_flag,
                                                            int* __restrict__ ws, int64_t ws_ints) {
  __shared__ uint32_t s_prefix;
  __shared__ int s_above;
  __shared__ int lds4[4];
  const int b = blockIdx.y;
  int* w = ws + b * ws_ints;
  const int tid = threadIdx.x;
  if (tid < 64)
    fv_select(w + 3 * 256, static_cast<uint32_t>(w[kASel + 12]), w[kASel + 13], removed, 0, &s_prefix,
              &s_above);
  __syncthreads();
  const uint32_t thresh = s_prefix;
  if (blockIdx.x == 0 && tid == 0) {
    w[kASel + 16] = static_cast<int>(thresh);
    w[kASel + 17] = removed - s_above;  // ties to remove, lowest position first
  }
  const float* bb = best + static_cast<int64_t>(b) * ns;
  int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  uint8_t* flag = removed_flag + static_cast<int64_t>(b) * ns;
  const int i0 = blockIdx.x * kAChunk + tid * kAPer;
  int ties = 0;
#pragma unroll
  for (int k = 0; k < kAPer; ++k) {
    const int i = i0 + k;
    if (i < ns) {
      const uint32_t key = ord32(bb[i]);
      const bool rm = key > thresh;
      flag[i] = rm ? 1 : 0;
      ties += key == thresh;
      if (rm) {
        const int64_t sid = source_ids[i];
        if (sid >= 0 && sid < total) inv[sid] = -1;
      }
    }
  }
  int n = 0;
  scan256(ties, lds4, &n);
  if (tid == 0) w[kAGroupsAt + blockIdx.x] = n;
}

__global__ __launch_bounds__(kAThreads) void fva_ties_kernel(const float* __restrict__ best,
                                                            const int64_t* __restrict__ source_ids,
                                                            int ns, int total,
                                                            int64_t* __restrict__ inverse,
                                                            uint8_t* __restrict__ removed_flag,
                                                            const int* __restrict__ ws, int64_t ws_ints) {
  __shared__ int lds4[4];
  const int b = blockIdx.y;
  const int* w = ws + b * ws_ints;
  const int tid = threadIdx.x;
  const uint32_t thresh = static_cast<uint32_t>(w[kASel + 16]);
  const int need = w[kASel + 17];
  int before = 0;  // ties in earlier groups
  for (int g = tid; g < static_cast<int>(blockIdx.x); g += kAThreads) before += w[kAGroupsAt + g];
  int sum = 0;
  scan256(before, lds4, &sum);
  before = sum;
  if (before >= need) return;  // uniform
  const float* bb = best + static_cast<int64_t>(b) * ns;
  int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  uint8_t* flag = removed_flag + static_cast<int64_t>(b) * ns;
  const int i0 = blockIdx.x * kAChunk + tid * kAPer;
  uint32_t tie_bits = 0;
#pragma unroll
  for (int k = 0; k < kAPer; ++k) {
    const int i = i0 + k;
    tie_bits |= (i < ns && ord32(bb[i]) == thresh ? 1u : 0u) << k;
  }
  int n = 0;
  int rank = before + scan256(__popc(tie_bits), lds4, &n);
#pragma unroll
  for (int k = 0; k < kAPer; ++k) {
    if ((tie_bits >> k) & 1u) {
      if (rank < need) {
        const int i = i0 + k;
        flag[i] = 1;
        const int64_t sid = source_ids[i];
        if (sid >= 0 && sid < total) inv[sid] = -1;
      }
      ++rank;
    }
  }
}

__global__ __launch_bounds__(kAThreads) void fva_kcount_kernel(int total, const int64_t* __restrict__ inverse,
                                                              int* __restrict__ ws, int64_t ws_ints,
                                                              int s_groups) {
  __shared__ int lds4[4];
  const int b = blockIdx.y;
  const int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  const int t0 = blockIdx.x * kAChunk + threadIdx.x * kAPer;
  int kept = 0;
#pragma unroll
  for (int k = 0; k < kAPer; ++k) kept += (t0 + k < total && inv[t0 + k] == 0) ? 1 : 0;
  int n = 0;
  scan256(kept, lds4, &n);
  if (threadIdx.x == 0) ws[b * ws_ints + kAGroupsAt + s_groups + blockIdx.x] = n;
}

__global__ __launch_bounds__(kAThreads) void fva_compact_kernel(int total, int removed,
                                                               int64_t* __restrict__ inverse,
                                                               int64_t* __restrict__ keep,
                                                               const int* __restrict__ ws, int64_t ws_ints,
                                                               int s_groups) {
  __shared__ int lds4[4];
  const int b = blockIdx.y;
  const int* w = ws + b * ws_ints + kAGroupsAt + s_groups;
  const int tid = threadIdx.x;
  int before = 0;
  for (int g = tid; g < static_cast<int>(blockIdx.x); g += kAThreads) before += w[g];
  int sum = 0;
  scan256(before, lds4, &sum);
  int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  int64_t* kp = keep + static_cast<int64_t>(b) * (total - removed);
  const int t0 = blockIdx.x * kAChunk + tid * kAPer;
  uint32_t kept_bits = 0;
#pragma unroll
  for (int k = 0; k < kAPer; ++k) kept_bits |= (t0 + k < total && inv[t0 + k] == 0 ? 1u : 0u) << k;
  int n = 0;
  int rank = sum + scan256(__popc(kept_bits), lds4, &n);
  const int n_keep = total - removed;
#pragma unroll
  for (int k = 0; k < kAPer; ++k) {
    if ((kept_bits >> k) & 1u) {
      inv[t0 + k] = rank;
      if (rank < n_keep) kp[rank] = t0 + k;  // always true for a valid (disjoint) source list
      ++rank;
    }
  }
}

__global__ __launch_bounds__(kAThreads) void fva_inverse_kernel(const int32_t* __restrict__ target,
                                                               const int64_t* __restrict__ source_ids,
                                                               const int64_t* __restrict__ dest_ids,
                                                               int ns, int nd, int total,
                                                               int64_t* __restrict__ inverse,
                                                               const uint8_t* __restrict__ removed_flag) {
  const int b = blockIdx.y;
  const int32_t* tb = target + static_cast<int64_t>(b) * ns;
  int64_t* inv = inverse + static_cast<int64_t>(b) * total;
  const uint8_t* flag = removed_flag + static_cast<int64_t>(b) * ns;
  const int i0 = blockIdx.x * kAChunk + threadIdx.x * kAPer;
  int64_t sid[kAPer], dst[kAPer];
#pragma unroll
  for (int k = 0; k < kAPer; ++k) {
    const int i = i0 + k;
    sid[k] = -1;
    dst[k] = -1;
    if (i < ns && flag[i]) {
      sid[k] = source_ids[i];
      const int32_t d = tb[i];
      dst[k] = (d >= 0 && d < nd) ? dest_ids[d] : -1;
    }
  }
#pragma unroll
  for (int k = 0; k < kAPer; ++k)
    if (sid[k] >= 0 && sid[k] < total) inv[sid[k]] = (dst[k] >= 0 && dst[k] < total) ? inv[dst[k]] : -1;
}

// ---------------------------------------------------------------------------
// A whole FastVGGT plan of one batch element in one launch of one work-group: the
// selection and keep / inverse above, the stable CSR of the clusters, their
// sizes and log sizes.  As launches these are twenty kernels, all latency: 28 us
// assembly, 24-31 us CSR and 8 us mass and int32 inverse at up to 12,288 tokens,
// and 3-4 us of host time for each.  Here every step between two barriers runs
// in one CU's LDS: 16 us at 1,044 tokens, 17 at 2,632, 31 at 8,528 (54 with
// every token on one destination).  Its time grows by 2 us per 1,024 tokens, the
// launches' hardly: 70 us against 73 at 20,580 tokens, 97 against 73 at 32,928,
// so larger plans take the launches.
//
//  * The removed-th largest key by binary search on its bits: a count per bit
//    is one ballot per 64 keys (held in registers), where a digit histogram
//    serialises on the few digits that bf16-rounded scores occupy.
//  * val[t] (u16): a kept token's compact id, a removed one's destination.
//  * Cluster order: block_csr.
// Results equal the launches' bit for bit.
constexpr int kPlanChunks = 12;                      // tokens <= 12 x 1024

struct PlanLds {
  int val_at, cnt_at, bits_at, bytes;  // byte offsets of val u16[total], cnt u16[kept + 2], removed bits
};
__host__ __device__ inline PlanLds plan_lds(int total, int kept) {
  PlanLds l;
  l.val_at = 0;
  l.cnt_at = (2 * total + 15) / 16 * 16;
  l.bits_at = l.cnt_at + (2 * (kept + 2) + 15) / 16 * 16;
  l.bytes = l.bits_at + (total + 31) / 32 * 4;
  return l;
}
constexpr int kPlanLds = 52 * 1024;  // >= plan_lds(kPlanChunks x kThreads, all of them kept).bytes
inline bool plan_fits(int64_t n_sources, int64_t total, int64_t removed) {
  return total <= kPlanChunks * kThreads && n_sources <= total && removed <= n_sources;
}

// C: chunks of 1,024 tokens (and of sources) the loops are unrolled for; a small plan's time is
// mostly the fetch of the code it runs through.
template <int C>
__global__ __launch_bounds__(kThreads) void fastvggt_plan_kernel(
    const float* __restrict__ best, const int32_t* __restrict__ target,
    const int64_t* __restrict__ source_ids, const int64_t* __restrict__ dest_ids, int ns, int nd, int total,
    int removed, int64_t* __restrict__ keep, int64_t* __restrict__ inverse, int32_t* __restrict__ inverse32,
    uint8_t* __restrict__ removed_flag, uint32_t* __restrict__ order, int32_t* __restrict__ offsets,
    float* __restrict__ mass, float* __restrict__ log_mass) {
  __shared__ __attribute__((aligned(16))) uint32_t state[kPlanLds / 4];
  __shared__ int counts[2][kWavesS];
  __shared__ int chunk_cnt[kPlanChunks * kWavesS];
  __shared__ BlockCsrLds<kPlanChunks> csr_lds;
  int* scan_lds = csr_lds.scan;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  const int kept = total - removed;
  const PlanLds at = plan_lds(total, kept);
  uint16_t* val = reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(state) + at.val_at);
  uint16_t* cnt = reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(state) + at.cnt_at);
  uint32_t* cnt32 = reinterpret_cast<uint32_t*>(cnt);
  uint32_t* bits = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(state) + at.bits_at);
  const int s_chunks = (ns + kThreads - 1) / kThreads;
  const int t_chunks = (total + kThreads - 1) / kThreads;

  for (int i = tid; i < (at.bytes - at.cnt_at) / 4; i += kThreads) cnt32[i] = 0;  // counters and bits

  // ---- keys; the removed-th largest of them.
  uint32_t key[C];  // 0 past the sources: below every key
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = c * kThreads + tid;
    key[c] = c < s_chunks && i < ns ? ord32(best[i]) : 0u;
  }
  int round = 0;
  auto count_from = [&](uint32_t bound) {  // keys >= bound (> 0), the same in every thread
    int n = 0;
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (c < s_chunks) n += __popcll(__ballot(key[c] >= bound));
    if (lane == 0) counts[round & 1][wave] = n;
    __syncthreads();
    int sum = 0;
#pragma unroll
    for (int w = 0; w < kWavesS; ++w) sum += counts[round & 1][w];
    ++round;
    return sum;
  };
  uint32_t thresh = 0;
  for (int bit = 31; bit >= 16; --bit)
    if (count_from(thresh | (1u << bit)) >= removed) thresh |= 1u << bit;
  // bf16 scores differ in the high half only (the low half of a negative one is all ones).
  if (count_from(thresh | 0xFFFFu) >= removed) {
    thresh |= 0xFFFFu;
  } else if (count_from(thresh | 1u) >= removed) {
    for (int bit = 15; bit >= 0; --bit)
      if (count_from(thresh | (1u << bit)) >= removed) thresh |= 1u << bit;
  }
  const int need_ties = removed - (thresh == 0xFFFFFFFFu ? 0 : count_from(thresh + 1));

  // ---- ranks of the ties, in source order.
  // In-place exclusive scan of chunk_cnt[0, chunks x waves) -> each (chunk, wave)'s base.
  auto scan_chunks = [&](int chunks) {
    __syncthreads();
    static_assert(kPlanChunks * kWavesS <= kThreads, "one count per thread");
    const int n = chunks * kWavesS;
    int sum = 0;
    const int mine = tid < n ? chunk_cnt[tid] : 0;
    const int pre = block_exclusive_scan(mine, scan_lds, &sum);
    if (tid < n) chunk_cnt[tid] = pre;
    __syncthreads();
  };
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (c < s_chunks) {
      const uint64_t m = __ballot(key[c] == thresh);
      if (lane == 0) chunk_cnt[c * kWavesS + wave] = __popcll(m);
    }
  scan_chunks(s_chunks);
  // ---- removed sources and their destinations (0xFFFF: not a token).  Four chunks' ids are
  // loaded together, whether their sources are removed or not.
#pragma unroll
  for (int c0 = 0; c0 < C; c0 += 4)
    if (c0 < s_chunks) {
      int64_t sid[4], dst[4];
      int32_t d[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = min((c0 + q) * kThreads + tid, ns - 1);
        sid[q] = source_ids[i];
        d[q] = target[i];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool ok = d[q] >= 0 && d[q] < nd;
        dst[q] = nd > 0 ? dest_ids[ok ? d[q] : 0] : -1;
        if (!ok || dst[q] < 0 || dst[q] >= total) dst[q] = 0xFFFF;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = c0 + q;
        if (c >= s_chunks) continue;
        const int i = c * kThreads + tid;
        const uint64_t m = __ballot(key[c] == thresh);
        const int rank = chunk_cnt[c * kWavesS + wave] + __popcll(m & below);
        const bool rm = i < ns && (key[c] > thresh || (key[c] == thresh && rank < need_ties));
        if (i < ns) removed_flag[i] = rm ? 1 : 0;
        if (rm && sid[q] >= 0 && sid[q] < total) {
          atomicOr(&bits[sid[q] >> 5], 1u << (sid[q] & 31));
          val[sid[q]] = static_cast<uint16_t>(dst[q]);
        }
      }
    }
  __syncthreads();

  // ---- compact ids of the kept tokens, ascending; the keep list.
  auto is_removed = [&](int t) { return ((bits[t >> 5] >> (t & 31)) & 1u) != 0u; };
  for (int c = 0; c < t_chunks; ++c) {
    const int t = c * kThreads + tid;
    const uint64_t m = __ballot(t < total && !is_removed(t));
    if (lane == 0) chunk_cnt[c * kWavesS + wave] = __popcll(m);
  }
  scan_chunks(t_chunks);
  for (int c = 0; c < t_chunks; ++c) {
    const int t = c * kThreads + tid;
    const bool k = t < total && !is_removed(t);
    const uint64_t m = __ballot(k);
    const int rank = chunk_cnt[c * kWavesS + wave] + __popcll(m & below);
    if (k) {
      val[t] = static_cast<uint16_t>(rank);
      if (rank < kept) keep[rank] = t;  // always true for a valid (disjoint) source list
    }
  }
  __syncthreads();

  // ---- inverse, and every token's cluster and slot in it (a token without one: cluster `kept`).
  uint32_t place[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int t = c * kThreads + tid;
    place[c] = 0;
    if (c < t_chunks && t < total) {
      int k = val[t];
      if (is_removed(t)) k = k == 0xFFFF || is_removed(k) ? -1 : val[k];
      if (k >= kept) k = -1;
      inverse[t] = k;
      inverse32[t] = k;
      place[c] = take_place(cnt32, k < 0 ? kept : k);
    }
  }
  __syncthreads();
  // val's space holds the members from here on.
  block_csr<C>(
      place, total, kept, val, cnt, csr_lds, order, offsets, [&](int k, int size) {
        const float m = static_cast<float>(size);
        mass[k] = m;
        log_mass[k] = logf(m);
      });
}

}  // namespace
}  // namespace vgo

extern "C" int vgo_fastvggt_plan_fits(int64_t n_sources, int64_t total_tokens, int64_t removed) {
  return n_sources >= 1 && removed >= 1 && vgo::plan_fits(n_sources, total_tokens, removed) ? 1 : 0;
}

extern "C" int vgo_fastvggt_plan(const float* best, const int32_t* target, const int64_t* source_ids,
                                 const int64_t* dest_ids, int64_t n_sources, int64_t n_dest,
                                 int64_t total_tokens, int64_t removed, int64_t* keep, int64_t* inverse,
                                 int32_t* inverse32, uint8_t* removed_flag, uint32_t* order,
                                 int32_t* offsets, float* mass, float* log_mass, void* stream) {
  using namespace vgo;
  VGO_REQUIRE(n_sources >= 0 && n_dest >= 0 && total_tokens >= 0, "fastvggt_plan: negative size");
  VGO_REQUIRE(removed >= 1 && removed <= n_sources, "fastvggt_plan: removed must lie in [1, sources]");
  VGO_REQUIRE(n_sources + n_dest <= total_tokens && total_tokens < (1LL << 30),
              "fastvggt_plan: inconsistent token counts");
  VGO_REQUIRE(best && target && source_ids && dest_ids && keep && inverse && inverse32 && removed_flag && order &&
                  offsets && mass && log_mass,
              "fastvggt_plan: null pointer");
  if (!plan_fits(n_sources, total_tokens, removed))
    return fail(VGO_EUNSUPPORTED, "fastvggt_plan: too many tokens for one work-group");
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kThreads), 0, as_stream(stream), best, target, source_ids, dest_ids,
                       static_cast<int>(n_sources), static_cast<int>(n_dest), static_cast<int>(total_tokens),
                       static_cast<int>(removed), keep, inverse, inverse32, removed_flag, order, offsets, mass,
                       log_mass);
  };
  if (total_tokens <= 4 * kThreads)
    launch(fastvggt_plan_kernel<4>);
  else
    launch(fastvggt_plan_kernel<kPlanChunks>);
  return check_launch("fastvggt_plan");
}

extern "C" int vgo_fastvggt_assemble(const float* best, const int32_t* target,
                                     const int64_t* source_ids, const int64_t* dest_ids,
                                     int64_t batch, int64_t n_sources, int64_t n_dest,
                                     int64_t total_tokens, int64_t removed, int64_t* keep,
                                     int64_t* inverse, uint8_t* removed_flag, void* stream) {
  using namespace vgo;
  VGO_REQUIRE(batch >= 0 && n_sources >= 0 && n_dest >= 0 && total_tokens >= 0,
              "fastvggt_assemble: negative size");
  VGO_REQUIRE(removed >= 1 && removed <= n_sources, "fastvggt_assemble: removed must lie in [1, sources]");
  VGO_REQUIRE(n_sources + n_dest <= total_tokens && total_tokens < (1LL << 30),
              "fastvggt_assemble: inconsistent token counts");
  if (batch == 0) return VGO_OK;
  VGO_REQUIRE(best && target && source_ids && dest_ids && keep && inverse && removed_flag,
              "fastvggt_assemble: null pointer");
  hipLaunchKernelGGL(fastvggt_assemble_kernel, dim3(static_cast<unsigned>(batch)), dim3(kThreads),
                     0, as_stream(stream), best, target, source_ids, dest_ids,
                     static_cast<int>(n_sources), static_cast<int>(n_dest),
                     static_cast<int>(total_tokens), static_cast<int>(removed), keep, inverse,
                     removed_flag);
  return check_launch("fastvggt_assemble");
}

extern "C" int vgo_sparse_convex_assemble(const float* fit, const float* alpha, const int64_t* support,
                                          const int64_t* candidate, const float* top1,
                                          float easy_threshold, const int* failed_count,
                                          int64_t n_candidates, int64_t total_tokens, float threshold,
                                          int64_t* keep, int64_t* original_to_compact, int64_t* source,
                                          int64_t* parent, float* weight, float* stats, void* stream) {
  using namespace vgo;
  VGO_REQUIRE(n_candidates >= 0 && total_tokens >= n_candidates && total_tokens < (1LL << 30),
              "sparse_convex_assemble: bad size");
  VGO_REQUIRE(keep && original_to_compact && stats, "sparse_convex_assemble: null pointer");
  VGO_REQUIRE(n_candidates == 0 || (fit && alpha && support && candidate && source && parent && weight),
              "sparse_convex_assemble: null pointer");
  const int n = static_cast<int>(n_candidates), total = static_cast<int>(total_tokens);
  hipLaunchKernelGGL(sparse_convex_select_kernel, dim3(1), dim3(kThreads), 0, as_stream(stream), fit, candidate, top1,
                     easy_threshold, failed_count, n, total, threshold, original_to_compact, parent, stats);
  const int64_t items = 4 * n_candidates > total_tokens ? 4 * n_candidates : total_tokens;
  if (items > 0) {
    hipLaunchKernelGGL(sparse_convex_fill_kernel, dim3(static_cast<unsigned>((items + 255) / 256)), dim3(256), 0,
                       as_stream(stream), alpha, support, candidate, original_to_compact, stats, n, total, keep,
                       source, parent, weight);
  }
  return check_launch("sparse_convex_assemble");
}

extern "C" int vgo_fastvggt_assemble_workspace(int64_t batch, int64_t n_sources, int64_t total_tokens,
                                               size_t* bytes) {
  using namespace vgo;
  VGO_REQUIRE(bytes, "fastvggt_assemble: null size pointer");
  VGO_REQUIRE(batch >= 0 && n_sources >= 0 && total_tokens >= 0 && total_tokens < (1LL << 30),
              "fastvggt_assemble: bad size");
  const int s_groups = static_cast<int>((n_sources + kAChunk - 1) / kAChunk);
  const int t_groups = static_cast<int>((total_tokens + kAChunk - 1) / kAChunk);
  *bytes = static_cast<size_t>(batch) * fv_ws_ints(s_groups, t_groups) * sizeof(int);
  return VGO_OK;
}

extern "C" int vgo_fastvggt_assemble_ws(const float* best, const int32_t* target,
                                        const int64_t* source_ids, const int64_t* dest_ids,
                                        int64_t batch, int64_t n_sources, int64_t n_dest,
                                        int64_t total_tokens, int64_t removed, int64_t* keep,
                                        int64_t* inverse, uint8_t* removed_flag, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  using namespace vgo;
  VGO_REQUIRE(batch >= 0 && n_sources >= 0 && n_dest >= 0 && total_tokens >= 0,
              "fastvggt_assemble: negative size");
  VGO_REQUIRE(removed >= 1 && removed <= n_sources, "fastvggt_assemble: removed must lie in [1, sources]");
  VGO_REQUIRE(n_sources + n_dest <= total_tokens && total_tokens < (1LL << 30),
              "fastvggt_assemble: inconsistent token counts");
  VGO_REQUIRE(batch <= 0xffff, "fastvggt_assemble: batch too large");
  if (batch == 0) return VGO_OK;
  VGO_REQUIRE(best && target && source_ids && dest_ids && keep && inverse && removed_flag,
              "fastvggt_assemble: null pointer");
  const int ns = static_cast<int>(n_sources), total = static_cast<int>(total_tokens);
  const int s_groups = (ns + kAChunk - 1) / kAChunk;
  const int t_groups = (total + kAChunk - 1) / kAChunk;
  const int64_t ws_ints = fv_ws_ints(s_groups, t_groups);
  if (workspace == nullptr ||
      workspace_bytes < static_cast<size_t>(batch) * ws_ints * sizeof(int))
    return fail(VGO_EWORKSPACE, "fastvggt_assemble: workspace too small");
  VGO_REQUIRE(aligned(workspace, 4), "fastvggt_assemble: workspace must be 4-byte aligned");
  int* ws = static_cast<int*>(workspace);
  hipStream_t s = as_stream(stream);
  const unsigned nb = static_cast<unsigned>(batch);
  hipLaunchKernelGGL(fva_init_kernel, dim3(t_groups, nb), dim3(kAThreads), 0, s, total, inverse, ws, ws_ints);
  for (int pass = 0; pass < 4; ++pass)
    hipLaunchKernelGGL(fva_hist_kernel, dim3(s_groups, nb), dim3(kAThreads), 0, s, best, ns,
                       static_cast<int>(removed), pass, ws, ws_ints);
  hipLaunchKernelGGL(fva_mark_kernel, dim3(s_groups, nb), dim3(kAThreads), 0, s, best, source_ids, ns, total,
                     static_cast<int>(removed), inverse, removed_flag, ws, ws_ints);
  hipLaunchKernelGGL(fva_ties_kernel, dim3(s_groups, nb), dim3(kAThreads), 0, s, best, source_ids, ns, total,
                     inverse, removed_flag, ws, ws_ints);
  hipLaunchKernelGGL(fva_kcount_kernel, dim3(t_groups, nb), dim3(kAThreads), 0, s, total, inverse, ws,
                     ws_ints, s_groups);
  hipLaunchKernelGGL(fva_compact_kernel, dim3(t_groups, nb), dim3(kAThreads), 0, s, total,
                     static_cast<int>(removed), inverse, keep, ws, ws_ints, s_groups);
  hipLaunchKernelGGL(fva_inverse_kernel, dim3(s_groups, nb), dim3(kAThreads), 0, s, target, source_ids,
                     dest_ids, ns, static_cast<int>(n_dest), total, inverse, removed_flag);
  return check_launch("fastvggt_assemble");
}
