// Mass-bias attention in fp32, O = softmax(Q K^T / sqrt(64) + log m) V, on the
// fp32 matrix instructions of gfx950 (the path outside autocast).
//
// Work of vggt_omega/models/mass_bias_attention.py:17-129 for fp32 inputs.
// Products and sums are fp32 throughout: v_mfma_f32_32x32x2_f32 multiplies and
// adds fp32 operands, at twice the rate of the vector unit's unpacked fmas and
// with one operand register per 2,048 multiply-adds.
//
// A task is 256 queries of one (batch, head), 4 waves x 64 queries (two
// 32-query column blocks).  Scores are computed transposed, S^T = K Q^T, so a
// lane owns one query per block and 16 of every 32 keys (register r of lane
// half h holds key 8 (r / 4) + 4 h + r % 4): the online softmax needs one
// exchange between the lane halves per 32 keys, and register r is already the
// B operand (k = lane half) of one step of O^T += V^T P^T, whose A operand is
// V[that key][d] read from a row-major V tile -- P is never moved.
// Keys stream through LDS in double-buffered tiles of 64 by LDS DMA (K rows
// XOR-permuted in 16-byte chunks so that 32 rows read at one chunk fall in
// distinct banks; V rows are read along d and need no permutation).
//
// Rounding: a 32-key chunk's P and P V are summed on their own (P V from a zero
// accumulator) and then join the running sums with one fma each, so the
// rounding of the sums grows with sqrt(32) + sqrt(nk / 32), not sqrt(nk).
//
// Bound: the matrix pipe (128 MFMAs of 64 cycles per wave and 64 queries x 32
// keys; two waves per SIMD, one's softmax under the other's MFMAs).  Measured,
// 16 heads x 4,111 queries x 2,057 keys: 326 us, 106 TFLOP/s (0.68 of the 157
// TFLOP/s fp32 matrix peak) against 6,546 us for one query per lane on the
// vector unit (1,040 single-wave groups, K and V broadcast from LDS per
// multiply); relative error against 64 bits 3.5e-7 (3.8e-7 before).
#include <algorithm>

#include "attention_f32.h"

namespace vgo {
namespace {

constexpr int kD = 64;
constexpr int kKeys = 64;      // keys per LDS tile
constexpr int kChunk = 32;     // keys whose P and P V are summed on their own
constexpr int kWaves = 4;
constexpr int kQWave = 64;     // queries per wave
constexpr int kQTask = kWaves * kQWave;
constexpr int kTile = kKeys * kD;
constexpr float kLog2e = 1.4426950408889634f;
// Partial state of a task cut between work-groups: O [256][64], m [256], l [256].
constexpr int64_t kPartialFloats = kQTask * (kD + 2);
constexpr int kGroupsPerCu = 2;
// Key tiles per work-group, at least: below this the partial state it would
// write (66 KB) costs more than the tile it takes off another work-group.
constexpr int64_t kMinUnits = 2;

struct Args {
  const float* q;
  const float* k;
  const float* v;
  const float* bias;
  float* out;
  int heads, nq, nk, n_qblocks, ntiles;
  int64_t qsb, qsh, qsn, ksb, ksh, ksn, vsb, vsh, vsn, osb, osh, osn;
  // Split evenly over `groups` work-groups: the (task, key tile) units or, without partial states,
  // whole tasks.
  int64_t units;
  int tasks, groups;
  float* partial;  // two states per work-group
};

// LDS position of element d of K row `row`: 16-byte chunks XOR-permuted by row & 15.
__device__ __forceinline__ int k_chunk(int row, int chunk) { return row * kD + ((chunk ^ (row & 15)) << 2); }

template <bool kVec>
struct Segment {
  const Args& a;
  float* k_lds;  // [2][kTile]
  float* v_lds;  // [2][kTile]
  float* b_lds;  // [2][kKeys]
  int tid, wave, lane, l32, hh;
  const float* kp;
  const float* vp;

  // Key tile t into buffer buf.  kVec: by LDS DMA (rows past n_key read the last
  // key; fix_tail then removes them), to be waited for with wait_vmem<0>.
  __device__ __forceinline__ void stage(int t, int buf) const {
    const int kt = t * kKeys;
    if constexpr (kVec) {
      const float* kb = kp + static_cast<int64_t>(kt) * a.ksn;
      const float* vb = vp + static_cast<int64_t>(kt) * a.vsn;
      const int last = a.nk - 1 - kt;
      if (a.bias != nullptr && wave == 0)
        lds_dma4(a.bias + kt, static_cast<uint32_t>(min(lane, last)) * 4u, lds_offset(b_lds + buf * kKeys));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r0 = (wave * 4 + i) * 4;
        const int row = r0 + (lane >> 4);
        const uint32_t src = static_cast<uint32_t>(min(row, last));
        const uint32_t kc = ((lane & 15) ^ (row & 15)) * 16u;
        lds_dma16(kb, src * static_cast<uint32_t>(a.ksn) * 4u + kc, lds_offset(k_lds + buf * kTile + r0 * kD));
        lds_dma16(vb, src * static_cast<uint32_t>(a.vsn) * 4u + (lane & 15) * 16u,
                  lds_offset(v_lds + buf * kTile + r0 * kD));
      }
    } else {
      for (int i = tid; i < kTile; i += kWaves * 64) {
        const int row = i / kD, d = i % kD;
        const bool ok = kt + row < a.nk;
        k_lds[buf * kTile + k_chunk(row, d >> 2) + (d & 3)] = ok ? kp[(kt + row) * a.ksn + d] : 0.0f;
        v_lds[buf * kTile + i] = ok ? vp[(kt + row) * a.vsn + d] : 0.0f;
      }
      if (tid < kKeys && a.bias != nullptr) b_lds[buf * kKeys + tid] = kt + tid < a.nk ? a.bias[kt + tid] : 0.0f;
    }
  }

  // Rows past n_key of the last tile: weight 0 (bias -inf) and zero values.
  __device__ __forceinline__ void fix_tail(int t, int buf) const {
    const int valid = a.nk - t * kKeys;
    for (int i = valid * kD + tid; i < kTile; i += kWaves * 64) v_lds[buf * kTile + i] = 0.0f;
    if (tid >= valid && tid < kKeys) b_lds[buf * kKeys + tid] = -__builtin_inff();
  }
};

// The wave's QB query blocks: Q operands, running max / sum and O^T.
template <int QB>
struct Wave {
  float q[QB][kD / 2];  // q[8j + 4 (lane / 32) + e] at [4j + e]
  float m[QB], l[QB];
  f32x16 o[QB][2];

  template <bool kVec>
  __device__ __forceinline__ void init(const float* qp, int64_t qsn, int q0, int nq, int l32, int hh) {
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const float* row = qp + static_cast<int64_t>(min(q0 + 32 * b + l32, nq - 1)) * qsn;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (kVec) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(row + 8 * j + 4 * hh);
#pragma unroll
          for (int e = 0; e < 4; ++e) q[b][4 * j + e] = x[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) q[b][4 * j + e] = row[8 * j + 4 * hh + e];
        }
      }
      m[b] = -__builtin_inff();
      l[b] = 0.0f;
      o[b][0] = o[b][1] = f32x16{};
    }
  }

  // One 32-key chunk of a tile: kl / vl / bl point at its first row.
  __device__ __forceinline__ void chunk(const float* kl, const float* vl, const float* bl, int l32, int hh) {
    f32x16 s[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) s[b] = f32x16{};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 kx = *reinterpret_cast<const f32x4*>(kl + k_chunk(l32, 2 * j + hh));
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < QB; ++b)
          s[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[e], q[b][4 * j + e], s[b], 0, 0, 0);
    }
    f32x4 bias[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bias[g] = *reinterpret_cast<const f32x4*>(bl + 8 * g + 4 * hh);
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[g][e] *= kLog2e;
    }
    constexpr float kScaleLog2 = 0.125f * kLog2e;
    float corr[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float mx = -__builtin_inff();
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[b][r] = fmaf(s[b][r], kScaleLog2, bias[r >> 2][r & 3]);
        mx = fmaxf(mx, s[b][r]);
      }
      const float mnew = fmaxf(m[b], half_max(mx));
      // No finite logit yet (every key so far of mass 0): every P is 0 and the
      // sums stay 0, where -inf - -inf would make them NaN.
      const float base = mnew == -__builtin_inff() ? 0.0f : mnew;
      corr[b] = __builtin_amdgcn_exp2f(m[b] - base);
      float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[b][r] = __builtin_amdgcn_exp2f(s[b][r] - base);
        part[r & 3] += s[b][r];
      }
      l[b] = fmaf(l[b], corr[b], (part[0] + part[1]) + (part[2] + part[3]));
      m[b] = mnew;
    }
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
      f32x16 t[QB];
#pragma unroll
      for (int b = 0; b < QB; ++b) t[b] = f32x16{};
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float vx = vl[(8 * (r >> 2) + 4 * hh + (r & 3)) * kD + 32 * dt + l32];
#pragma unroll
        for (int b = 0; b < QB; ++b) t[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx, s[b][r], t[b], 0, 0, 0);
      }
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][dt][r] = fmaf(o[b][dt][r], corr[b], t[b][r]);
    }
  }

  // The finished rows, or (state != null) the wave's part of a partial state.
  template <bool kVec>
  __device__ __forceinline__ void store(float* op, int64_t osn, float* state, int q_task, int q_wave, int nq,
                                        int l32, int hh) {
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const int local = q_wave + 32 * b + l32;
      const float total = half_sum(l[b]);
      if (q_task + local >= nq) continue;
      if (state != nullptr) {
        float* dst = state + local * kD;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * g + 4 * hh) =
                f32x4{o[b][dt][4 * g], o[b][dt][4 * g + 1], o[b][dt][4 * g + 2], o[b][dt][4 * g + 3]};
        if (hh == 0) {
          state[kQTask * kD + local] = m[b];
          state[kQTask * (kD + 1) + local] = total;
        }
        continue;
      }
      float* dst = op + static_cast<int64_t>(q_task + local) * osn;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = o[b][dt][4 * g + e] / total;
          if constexpr (kVec) {
            *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * g + 4 * hh) = x;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[32 * dt + 8 * g + 4 * hh + e] = x[e];
          }
        }
    }
  }
};

// Key tiles [t0, t1) of one task.  QB: query blocks of this wave (0: it only
// stages tiles and meets the barriers).
template <bool kVec, int QB>
__device__ __forceinline__ void run_tiles(const Segment<kVec>& sg, const float* qp, float* op, float* state,
                                          int q_task, int t0, int t1) {
  const Args& a = sg.a;
  const int q_wave = sg.wave * kQWave;
  Wave<QB == 0 ? 1 : QB> w;
  if constexpr (QB > 0) w.template init<kVec>(qp, a.qsn, q_task + q_wave, a.nq, sg.l32, sg.hh);
  sg.stage(t0, 0);
  wait_vmem<0>();
  __syncthreads();
  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1;
    if ((t + 1) * kKeys > a.nk) {  // the same for every wave
      sg.fix_tail(t, buf);
      __syncthreads();
    }
    if (t + 1 < t1) sg.stage(t + 1, buf ^ 1);
    if constexpr (QB > 0) {
#pragma unroll 1
      for (int c = 0; c < kKeys / kChunk; ++c)
        w.chunk(sg.k_lds + buf * kTile + c * kChunk * kD, sg.v_lds + buf * kTile + c * kChunk * kD,
                sg.b_lds + buf * kKeys + c * kChunk, sg.l32, sg.hh);
    }
    wait_vmem<0>();
    __syncthreads();
  }
  if constexpr (QB > 0) w.template store<kVec>(op, a.osn, state, q_task, q_wave, a.nq, sg.l32, sg.hh);
}

template <bool kVec>
__global__ __launch_bounds__(kWaves * 64, kGroupsPerCu) void attn_f32_kernel(const Args a) {
  __shared__ __attribute__((aligned(16))) float k_lds[2 * kTile];
  __shared__ __attribute__((aligned(16))) float v_lds[2 * kTile];
  __shared__ __attribute__((aligned(16))) float b_lds[2 * kKeys];
  const int w = xcd_remap(blockIdx.x, a.groups);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool cut = a.partial != nullptr;
  const int64_t u0 = cut ? sk_begin(w, a.units, a.groups) : sk_begin(w, a.tasks, a.groups) * a.ntiles;
  const int64_t u1 = cut ? sk_begin(w + 1, a.units, a.groups) : sk_begin(w + 1, a.tasks, a.groups) * a.ntiles;
  for (int64_t u = u0; u < u1;) {
    const int task = static_cast<int>(u / a.ntiles);
    const int t0 = static_cast<int>(u - static_cast<int64_t>(task) * a.ntiles);
    const int t1 = static_cast<int>(min(static_cast<int64_t>(a.ntiles), t0 + (u1 - u)));
    const int bh = task / a.n_qblocks;
    const int q_task = (task - bh * a.n_qblocks) * kQTask;
    const int b = bh / a.heads, h = bh - b * a.heads;
    // Biases: read by DMA with the tiles; without any, zeros (fix_tail may have
    // overwritten them in an earlier task).
    if (a.bias == nullptr && tid < 2 * kKeys) b_lds[tid] = 0.0f;
    const Segment<kVec> sg{a, k_lds, v_lds, b_lds, tid, wave, lane, lane & 31, lane >> 5,
                           a.k + b * a.ksb + h * a.ksh, a.v + b * a.vsb + h * a.vsh};
    const float* qp = a.q + b * a.qsb + h * a.qsh;
    float* op = a.out + b * a.osb + h * a.osh;
    // A cut task's state: slot 2w holds work-group w's first piece, 2w + 1 a later one.
    float* state = nullptr;
    if (t0 != 0 || t1 != a.ntiles) state = a.partial + (2 * static_cast<int64_t>(w) + (u != u0)) * kPartialFloats;
    const int left = a.nq - q_task - wave * kQWave;  // this wave's queries
    if (left > 32)
      run_tiles<kVec, 2>(sg, qp, op, state, q_task, t0, t1);
    else if (left > 0)
      run_tiles<kVec, 1>(sg, qp, op, state, q_task, t0, t1);
    else
      run_tiles<kVec, 0>(sg, qp, op, state, q_task, t0, t1);
    u += t1 - t0;
  }
}

// Combines the partial states of the tasks that were cut: 16 rows per block.
constexpr int kMergeRows = 16;
template <bool kVec>
__global__ __launch_bounds__(256) void attn_f32_merge_kernel(const Args a) {
  constexpr int kParts = kQTask / kMergeRows;
  const int task = blockIdx.x / kParts;
  const int local = (blockIdx.x % kParts) * kMergeRows + (threadIdx.x >> 4);
  const int d = (threadIdx.x & 15) * 4;
  const int64_t first = static_cast<int64_t>(task) * a.ntiles;
  const int64_t w0 = sk_owner(first, a.units, a.groups);
  const int64_t w1 = sk_owner(first + a.ntiles - 1, a.units, a.groups);
  if (w0 == w1) return;  // one work-group ran the whole task
  const int bh = task / a.n_qblocks;
  const int row = (task - bh * a.n_qblocks) * kQTask + local;
  if (row >= a.nq) return;
  auto state = [&](int64_t w) {
    const bool later = w == w0 && sk_begin(w, a.units, a.groups) < first;
    return a.partial + (2 * w + (later ? 1 : 0)) * kPartialFloats;
  };
  float m = -__builtin_inff();
  for (int64_t w = w0; w <= w1; ++w) m = fmaxf(m, state(w)[kQTask * kD + local]);
  const float base = m == -__builtin_inff() ? 0.0f : m;
  float l = 0.0f;
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t w = w0; w <= w1; ++w) {
    const float* st = state(w);
    const float c = __builtin_amdgcn_exp2f(st[kQTask * kD + local] - base);
    l = fmaf(st[kQTask * (kD + 1) + local], c, l);
    const f32x4 x = *reinterpret_cast<const f32x4*>(st + local * kD + d);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(x[e], c, o[e]);
  }
  const int b = bh / a.heads, h = bh - b * a.heads;
  float* dst = a.out + b * a.osb + h * a.osh + static_cast<int64_t>(row) * a.osn + d;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = o[e] / l;
  if constexpr (kVec) {
    *reinterpret_cast<f32x4*>(dst) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[e] = o[e];
  }
}

int64_t tasks_of(const Problem& p) { return (p.nq + kQTask - 1) / kQTask * p.batch * p.heads; }
int64_t tiles_of(const Problem& p) { return (p.nk + kKeys - 1) / kKeys; }

// Tasks past this many rounds of the resident work-groups are not cut: the last round is then
// 1/64 of the time at most, and the merge would run 16 blocks for every task to find the few.
constexpr int64_t kMaxSplitRounds = 64;
// Work-groups of a launch without splitting.  A grid holds 2^32 threads; the tasks past that are
// second ones of a work-group.
constexpr int64_t kMaxGroups = int64_t{1} << 23;

// Work-groups over which the (task, key tile) units are split: two per CU, with
// at least kMinUnits tiles each.  0: not split, because the tasks already divide
// evenly over the resident work-groups, are more than the pieces, or are very many.
int64_t split_groups(const Problem& p) {
  const int64_t tasks = tasks_of(p), slots = int64_t{device_cus()} * kGroupsPerCu;
  if (tasks > kMaxSplitRounds * slots) return 0;
  const int64_t groups = std::min<int64_t>(slots, tasks * tiles_of(p) / kMinUnits);
  return groups > tasks || (groups == slots && tasks % groups != 0) ? groups : 0;
}

// 16-byte vector access (LDS DMA, Q loads, row stores): rows 16-byte aligned and
// a tile's row offsets within 32 bits.
bool vector_rows(const Problem& p) {
  for (const int64_t* s : {p.qs, p.ks, p.vs, p.os})
    for (int i = 0; i < 3; ++i)
      if (s[i] % 4 != 0) return false;
  const int64_t lim = int64_t{1} << 22;
  return aligned(p.q, 16) && aligned(p.k, 16) && aligned(p.v, 16) && aligned(p.out, 16) && p.ks[2] >= 0 &&
         p.ks[2] <= lim && p.vs[2] >= 0 && p.vs[2] <= lim;
}

}  // namespace

size_t attn_f32_workspace(const Problem& p) {
  return static_cast<size_t>(split_groups(p)) * 2 * kPartialFloats * sizeof(float);
}

int launch_attn_f32(const Problem& p, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  const int64_t tasks = tasks_of(p);
  VGO_REQUIRE(tasks <= 0x7fffffff, "mass_bias_attention: grid too large");
  Args a;
  a.q = static_cast<const float*>(p.q);
  a.k = static_cast<const float*>(p.k);
  a.v = static_cast<const float*>(p.v);
  a.bias = static_cast<const float*>(p.bias);
  a.out = static_cast<float*>(p.out);
  a.heads = static_cast<int>(p.heads);
  a.nq = static_cast<int>(p.nq);
  a.nk = static_cast<int>(p.nk);
  a.n_qblocks = static_cast<int>((p.nq + kQTask - 1) / kQTask);
  a.ntiles = static_cast<int>(tiles_of(p));
  a.qsb = p.qs[0], a.qsh = p.qs[1], a.qsn = p.qs[2];
  a.ksb = p.ks[0], a.ksh = p.ks[1], a.ksn = p.ks[2];
  a.vsb = p.vs[0], a.vsh = p.vs[1], a.vsn = p.vs[2];
  a.osb = p.os[0], a.osh = p.os[1], a.osn = p.os[2];
  a.units = tasks * a.ntiles;
  a.tasks = static_cast<int>(tasks);
  a.groups = static_cast<int>(std::min(tasks, kMaxGroups));
  a.partial = nullptr;
  const bool split = workspace != nullptr && workspace_bytes > 0 && workspace_bytes >= attn_f32_workspace(p);
  if (split) {
    a.groups = static_cast<int>(split_groups(p));
    a.partial = static_cast<float*>(workspace);
  }
  const bool vec = vector_rows(p);
  const dim3 grid(static_cast<unsigned>(a.groups)), block(kWaves * 64);
  if (vec)
    hipLaunchKernelGGL((attn_f32_kernel<true>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((attn_f32_kernel<false>), grid, block, 0, stream, a);
  const int status = check_launch("mass_bias_attention(f32)");
  if (status != VGO_OK || !split) return status;
  const dim3 merge_grid(static_cast<unsigned>(tasks * (kQTask / kMergeRows)));
  if (vec)
    hipLaunchKernelGGL((attn_f32_merge_kernel<true>), merge_grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((attn_f32_merge_kernel<false>), merge_grid, dim3(256), 0, stream, a);
  return check_launch("mass_bias_attention(f32 merge)");
}

}  // namespace vgo
