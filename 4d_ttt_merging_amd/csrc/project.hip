// Top-4 convex projection (unmerge), the restore step of a merge plan:
//   out[i,:] = sum_{c<4} w[i,c] * table[index[i,c],:]
//
// Work of vggt_omega/models/token_merging.py:387-414 (WeightedBilinearTokenPlan.
// restore: `parent = value[:, parent]; (parent * w.to(value.dtype)).sum(2)`) and
// :193-196 (TokenPlan.restore, the one-hot case).  The reference materialises
// [M,4,C] and sums it; here products are rounded to the value type exactly as
// the reference's elementwise multiply does and summed in fp32 in corner order.
//
// Bound: the gathers.  Four table rows per output row come from anywhere in the
// table, four times the bytes that are written, and whole-row gathers run at
// what the fabric behind the L2s gives (7 TB/s).  So the columns are cut into
// slices of W x 16 bytes, and each of the 8 XCDs takes its own slices over all
// rows: an XCD's 4 MB L2 then holds (part of) its slice of the table instead of
// an eighth of all whole-row gathers, and serves the repeats.  Index and weight
// are read once more per slice (32 B per row), which bounds W from below.
// Rows that share few table rows with others, or share them with their
// neighbours (restores of kept rows, one-hot maps, maps in locality order), gain
// nothing from the L2s' slices and pay for the repeated index: they are computed
// whole.  What a call's rows are like is in its index and weight, which the host
// does not read: the kernel takes a sample of them (sampled_kind).
#include <algorithm>
#include <type_traits>

#include "vgo_common.h"

namespace vgo {
namespace {

constexpr int kWaves = 4;  // waves per work-group

template <typename T>
struct Vec16;  // 16 bytes of T
template <>
struct Vec16<float> {
  typedef f32x4 type;
  static constexpr int n = 4;
};
template <>
struct Vec16<bf16_t> {
  typedef bf16x8 type;
  static constexpr int n = 8;
};
template <>
struct Vec16<f16_t> {
  typedef f16x8 type;
  static constexpr int n = 8;
};


// One output row's corners: the ids and weights, which of them are gathered
// (zero weights are not), and whether an id with a weight is out of range.
template <typename T>
struct Corners {
  i32x4 id;
  float w[4];
  bool use[4];
  bool bad;
  __device__ __forceinline__ void load(const int32_t* index, const float* weight, int64_t row,
                                       int64_t table_rows) {
    bad = false;
    id = i32x4{0, 0, 0, 0};
    f32x4 w4 = {0.0f, 0.0f, 0.0f, 0.0f};
    if (row >= 0) {
      id = *reinterpret_cast<const i32x4*>(index + 4 * row);
      w4 = *reinterpret_cast<const f32x4*>(weight + 4 * row);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      use[c] = w4[c] != 0.0f;
      if (use[c] && static_cast<uint32_t>(id[c]) >= static_cast<uint64_t>(table_rows)) {
        bad = true;
        use[c] = false;
      }
      w[c] = weight_as_value<T>(w4[c]);
    }
  }
  // 16 bytes of the output row from the corners' chunks.
  template <typename V>
  __device__ __forceinline__ V sum(const V (&y)[4]) const {
    constexpr int VN = Vec16<T>::n;
    float acc[VN];
#pragma unroll
    for (int j = 0; j < VN; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (use[c]) {
#pragma unroll
        for (int j = 0; j < VN; ++j) acc[j] = acc[j] + rounded_product<T>(to_f32(y[c][j]), w[c]);
      }
    }
    V o;
#pragma unroll
    for (int j = 0; j < VN; ++j) o[j] = from_f32<T>(bad ? __builtin_nanf("") : acc[j]);
    return o;
  }
};

// A unit is kRows = 2 * 64 / W output rows of one slice (W lanes of 16 bytes per
// row, two rows per lane, eight gathers in flight); units are ordered slice by
// slice, and XCD x (work-groups with blockIdx % 8 == x) runs the x-th eighth.
template <typename T, int W>
__device__ __forceinline__ void sliced_rows(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, const int32_t* __restrict__ order, T* __restrict__ out,
    int64_t out_stride, int64_t n_rows, int64_t table_rows, int dim, int groups) {
  const int n_slices = (dim + W * Vec16<T>::n - 1) / (W * Vec16<T>::n);
  typedef typename Vec16<T>::type V;
  constexpr int kGroup = 64 / W;
  constexpr int kRows = 2 * kGroup;
  const int lane = lane_id();
  const int xcd = blockIdx.x % kNumXcd;
  const int waves = groups / kNumXcd * kWaves;  // of this XCD
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) / kNumXcd * kWaves +
                                                  static_cast<int>(threadIdx.x >> 6));
  const int64_t blocks = (n_rows + kRows - 1) / kRows;  // units of one slice
  const int64_t units = blocks * n_slices;
  const int64_t u1 = units * (xcd + 1) / kNumXcd;
  for (int64_t u = units * xcd / kNumXcd + wave; u < u1; u += waves) {
    const int64_t slice = u / blocks;
    const int64_t r0 = (u - slice * blocks) * kRows + lane / W;
    const int64_t e = (slice * W + lane % W) * Vec16<T>::n;
    if (e >= dim) continue;
    Corners<T> corner[2];
    int64_t orow[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      // Output row of the work position: the position itself, or order[position]
      // (positions whose order entry is out of range produce nothing).
      const int64_t pos = r0 + r * kGroup;
      orow[r] = pos < n_rows ? pos : -1;
      if (order && orow[r] >= 0) {
        const int32_t o = order[pos];
        orow[r] = o >= 0 && o < n_rows ? o : -1;
      }
      corner[r].load(index, weight, orow[r], table_rows);
    }
    V y[2][4];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (corner[r].use[c])
          y[r][c] = *reinterpret_cast<const V*>(table + static_cast<int64_t>(corner[r].id[c]) * table_stride + e);
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (orow[r] >= 0)
        __builtin_nontemporal_store(corner[r].sum(y[r]), reinterpret_cast<V*>(out + orow[r] * out_stride + e));
  }
}

// Whole rows: each wave takes R consecutive output rows per step and issues the gathers of all
// of them (4 corners x CH 16-byte chunks per lane each) before reducing any.
//
// The loop of 1,048,576 rows over 65,536 of 1,024 channels in locality order (us, by slices and
// whole): bf16 1,660, 1,311; fp32 2,689, 2,439; one-hot rows 1,020, 615 and 1,919, 1,139.
//
// kRowSums (the gather probe, vgo_top4_gather_probe): each row's output values are summed in
// fp32 (per lane, then over the wave) and only that sum is written, to row_sums[row]: what the
// fabric gives random whole-row reads.
template <typename T, int R, int CH, bool kRowSums>
__device__ __forceinline__ void whole_rows(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, const int32_t* __restrict__ order, T* __restrict__ out,
    int64_t out_stride, int64_t n_rows, int64_t table_rows, int dim, int groups, float* __restrict__ row_sums) {
  typedef typename Vec16<T>::type V;
  constexpr int VN = Vec16<T>::n;
  const int lane = lane_id();
  const int64_t wave_gid = __builtin_amdgcn_readfirstlane(
      static_cast<int>(blockIdx.x) * kWaves + static_cast<int>(threadIdx.x >> 6));
  const int64_t step = static_cast<int64_t>(groups) * kWaves * R;
  for (int64_t r0 = wave_gid * R; r0 < n_rows; r0 += step) {
    Corners<T> corner[R];
    int64_t orow[R];
    float lane_sum[R];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      const int64_t pos = r0 + rr;
      orow[rr] = pos < n_rows ? pos : -1;
      if (order && orow[rr] >= 0) {
        const int32_t o = order[pos];
        orow[rr] = o >= 0 && o < n_rows ? o : -1;
      }
      lane_sum[rr] = 0.0f;
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) corner[rr].load(index, weight, orow[rr], table_rows);
    for (int base = 0; base < dim; base += CH * 64 * VN) {
      V y[R][CH][4];
#pragma unroll
      for (int rr = 0; rr < R; ++rr)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (corner[rr].use[c]) {
            const T* trow = table + static_cast<int64_t>(corner[rr].id[c]) * table_stride;
#pragma unroll
            for (int ch = 0; ch < CH; ++ch) {
              const int e = base + (ch * 64 + lane) * VN;
              if (e < dim) y[rr][ch][c] = *reinterpret_cast<const V*>(trow + e);
            }
          }
#pragma unroll
      for (int rr = 0; rr < R; ++rr) {
        if (orow[rr] < 0) continue;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) {
          const int e = base + (ch * 64 + lane) * VN;
          if (e >= dim) continue;
          const V o = corner[rr].sum(y[rr][ch]);
          if constexpr (kRowSums) {
#pragma unroll
            for (int j = 0; j < VN; ++j) lane_sum[rr] += to_f32(o[j]);
          } else {
            __builtin_nontemporal_store(o, reinterpret_cast<V*>(out + orow[rr] * out_stride + e));
          }
        }
      }
    }
    if constexpr (kRowSums) {
#pragma unroll
      for (int rr = 0; rr < R; ++rr) {
        float v = lane_sum[rr];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
        if (lane == 0 && orow[rr] >= 0) row_sums[orow[rr]] = v;
      }
    }
  }
}

// What the rows of a projection are like: one corner each (kept rows, one-hot maps), in a row with
// their neighbours or scattered; a part of them with one; four corners near each other (within a
// 32nd of the table); or four anywhere.
enum RowKind { kKept, kOneHot, kPart, kNear, kMixed, kKinds };
// Work-groups that compute rows of each kind whole; 0: by slices.
struct WholeRows {
  int groups[kKinds] = {};
};

// The kind of the rows, from 128 pairs of neighbours spread over the work positions: 8 KB that every
// work-group reads before it starts, so that all of them agree (within 1% of a call of 96 MB).  Only
// the time depends on it: a row has the same products and sums either way.
__device__ __forceinline__ RowKind sampled_kind(const int32_t* index, const float* weight, int64_t n_rows,
                                                int64_t table_rows) {
  constexpr int kSamples = kWaves * 64;
  __shared__ int counts[3][kWaves];
  const int t = static_cast<int>(threadIdx.x);
  const int64_t row = min(n_rows - 1, t / 2 * n_rows / (kSamples / 2) + (t & 1));
  const i32x4 id = *reinterpret_cast<const i32x4*>(index + 4 * row);
  const f32x4 w = *reinterpret_cast<const f32x4*>(weight + 4 * row);
  int used = 0, low = 0x7fffffff, high = -1;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (w[c] != 0.0f) {
      ++used;
      low = min(low, id[c]);
      high = max(high, id[c]);
    }
  }
  const int64_t close = table_rows / 32;
  const int64_t spread = static_cast<int64_t>(high) - low, step = static_cast<int64_t>(low) - __shfl_xor(low, 1);
  int sum = 0;
#pragma unroll
  for (int c = 1; c <= 4; ++c) sum += __popcll(__ballot(used >= c));
  const int together = __popcll(__ballot(used >= 2 && spread <= close));
  const int in_row = __popcll(__ballot(step >= -close && step <= close));
  if (lane_id() == 0) counts[0][t >> 6] = sum, counts[1][t >> 6] = together, counts[2][t >> 6] = in_row;
  __syncthreads();
  const auto total = [&](int i) { return counts[i][0] + counts[i][1] + counts[i][2] + counts[i][3]; };
  static_assert(kWaves == 4, "counts of four waves");
  if (2 * total(0) < 3 * kSamples) return 2 * total(2) > kSamples ? kKept : kOneHot;
  if (total(0) < 3 * kSamples) return kPart;
  return 2 * total(1) > kSamples ? kNear : kMixed;
}

template <typename T, int W>
__global__ __launch_bounds__(kWaves * 64) void top4_project_kernel(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, const int32_t* __restrict__ order, T* __restrict__ out,
    int64_t out_stride, int64_t n_rows, int64_t table_rows, int dim) {
  sliced_rows<T, W>(table, table_stride, index, weight, order, out, out_stride, n_rows, table_rows, dim, gridDim.x);
}

template <typename T, int R, int CH, bool kRowSums>
__global__ __launch_bounds__(kWaves * 64) void top4_rows_kernel(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, const int32_t* __restrict__ order, T* __restrict__ out,
    int64_t out_stride, int64_t n_rows, int64_t table_rows, int dim, float* __restrict__ row_sums) {
  whole_rows<T, R, CH, kRowSums>(table, table_stride, index, weight, order, out, out_stride, n_rows, table_rows,
                                 dim, gridDim.x, row_sums);
}

// Both, with the sampled rows deciding and each taking its number of the work-groups.  Whole rows
// have half the gathers of top4_rows_kernel in flight per wave (16 chunks), which keeps the kernel
// within the registers of five work-groups per CU that the slices need.
template <typename T, int W, int R, int CH>
__global__ __launch_bounds__(kWaves * 64, 5) void top4_sampled_kernel(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, T* __restrict__ out, int64_t out_stride, int64_t n_rows, int64_t table_rows,
    int dim, int slice_groups, WholeRows whole) {
  const RowKind kind = sampled_kind(index, weight, n_rows, table_rows);
  int groups = 0;
#pragma unroll
  for (int k = 0; k < kKinds; ++k) groups = kind == k ? whole.groups[k] : groups;
  if (groups > 0) {
    if (static_cast<int>(blockIdx.x) < groups)
      whole_rows<T, R, CH, false>(table, table_stride, index, weight, nullptr, out, out_stride, n_rows, table_rows,
                                  dim, groups, nullptr);
  } else if (static_cast<int>(blockIdx.x) < slice_groups) {
    sliced_rows<T, W>(table, table_stride, index, weight, nullptr, out, out_stride, n_rows, table_rows, dim,
                      slice_groups);
  }
}

// Fallback for rows whose byte size is not a multiple of 16: one element per lane.
template <typename T>
__global__ __launch_bounds__(256) void top4_project_scalar_kernel(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, const int32_t* __restrict__ order, T* __restrict__ out,
    int64_t out_stride, int64_t n_rows, int64_t pos0, int64_t table_rows, int dim) {
  const int64_t pos = pos0 + blockIdx.y;
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (pos >= n_rows || e >= dim) return;
  const int64_t row = order ? order[pos] : pos;
  if (row < 0 || row >= n_rows) return;
  float acc = 0.0f;
  bool bad = false;
  for (int c = 0; c < 4; ++c) {
    const float w = weight[4 * row + c];
    if (w == 0.0f) continue;
    const int32_t id = index[4 * row + c];
    if (static_cast<uint32_t>(id) >= static_cast<uint64_t>(table_rows)) {
      bad = true;
      continue;
    }
    acc = acc + (rounded_product<T>(to_f32(table[id * table_stride + e]),
                                            weight_as_value<T>(w)));
  }
  out[row * out_stride + e] = from_f32<T>(bad ? __builtin_nanf("") : acc);
}

// Operands of a launch of rows of whole 16-byte chunks (vector_rows).
template <typename T>
struct Rows {
  const T* table;
  int64_t table_stride;
  const int32_t* index;
  const float* weight;
  const int32_t* order;
  T* out;
  int64_t out_stride, n_rows, table_rows;
  int dim;
  hipStream_t stream;
  // 16-byte chunks per row per lane of a wave.
  int chunks() const { return (dim + 64 * Vec16<T>::n - 1) / (64 * Vec16<T>::n); }
  int64_t out_bytes() const { return n_rows * dim * static_cast<int64_t>(sizeof(T)); }
};

template <typename T, int W>
void launch_sliced(const Rows<T>& r, int groups_per_cu, const WholeRows& whole) {
  constexpr int kRows = 2 * 64 / W;
  const int64_t n_slices = (r.dim + W * Vec16<T>::n - 1) / (W * Vec16<T>::n);
  const int64_t units = (r.n_rows + kRows - 1) / kRows * n_slices;
  const int64_t per_xcd = (units + kNumXcd - 1) / kNumXcd;
  const int64_t cap = std::max<int64_t>(1, int64_t{device_cus()} * groups_per_cu / kNumXcd);
  const int groups = static_cast<int>(std::min<int64_t>(cap, (per_xcd + kWaves - 1) / kWaves)) * kNumXcd;
  const int most = *std::max_element(whole.groups, whole.groups + kKinds);
  if (most == 0) {
    hipLaunchKernelGGL((top4_project_kernel<T, W>), dim3(groups), dim3(kWaves * 64), 0, r.stream, r.table,
                       r.table_stride, r.index, r.weight, r.order, r.out, r.out_stride, r.n_rows, r.table_rows, r.dim);
    return;
  }
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(std::max(groups, most)), dim3(kWaves * 64), 0, r.stream, r.table, r.table_stride,
                       r.index, r.weight, r.out, r.out_stride, r.n_rows, r.table_rows, r.dim, groups, whole);
  };
  if (r.chunks() >= 4)
    launch(top4_sampled_kernel<T, W, 1, 4>);
  else
    launch(top4_sampled_kernel<T, W, 2, 2>);
}

// Whole rows: eight work-groups per CU, about 32 chunks (512 B) in flight per lane.
template <typename T, bool kRowSums>
void launch_rows(const Rows<T>& r, float* row_sums) {
  const int chunks = r.chunks(), rows_per_wave = chunks >= 4 ? 2 : chunks >= 2 ? 4 : 8;
  const int64_t need = (r.n_rows + kWaves * rows_per_wave - 1) / (kWaves * rows_per_wave);
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>(need, int64_t{device_cus()} * 8)));
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kWaves * 64), 0, r.stream, r.table, r.table_stride, r.index, r.weight,
                       r.order, r.out, r.out_stride, r.n_rows, r.table_rows, r.dim, row_sums);
  };
  if (chunks >= 4)
    launch(top4_rows_kernel<T, 2, 4, kRowSums>);
  else if (!kRowSums || chunks >= 2)
    launch(top4_rows_kernel<T, 4, 2, kRowSums>);
  else if constexpr (kRowSums)  // whole_rule leaves such short rows to the slices
    launch(top4_rows_kernel<T, 8, 1, true>);
}

template <typename T>
bool vector_rows(const void* table, int64_t table_stride, const void* out, int64_t out_stride, int64_t dim) {
  constexpr int VN = Vec16<T>::n;
  return dim % VN == 0 && table_stride % VN == 0 && out_stride % VN == 0 && aligned(table, 16) &&
         aligned(out, 16);
}

// Slice width and resident work-groups, measured over tables of 2,000 to 262,144
// rows of 768 and 1,024 channels, four times as many output rows (us; "whole":
// whole-row gathers):
//   bf16, 16,000 rows: 128 B slices 54, 512 B 65, whole 98; 65,536 rows: 304, 347,
//   384 (1,048,576 outputs: 1,179, 1,387, 1,471); 131,072: 709, 729, 755;
//   262,144: 1,555, 1,453, 1,512.
//   fp32, 16,000 rows: 256 B slices 78, 128 B 84, 512 B 117, whole 177; 65,536:
//   614, 662, 666, 749; 262,144: 2,883, 3,029, 3,418, 3,441.
// So 2-byte types take 128 B slices while the table's slice is at most three times
// an XCD's L2, then 512 B; fp32 (whose rows have twice the slices, each reading
// index and weight again) takes 256 B.  Four work-groups per CU keep the waves of
// an XCD closer to one slice than eight do (1,179 against 1,289 us at 65,536
// rows); where the slice is within half the L2 that does not matter and eight are
// faster in the 2-byte types (54 against 59 us at 16,000 rows, fp32 41 against 37
// at 8,000).
constexpr int64_t kNarrowRows = 98304;  // x 128 B = 12 MB
constexpr int64_t kHalfL2Rows = 16384;  // x 128 B = 2 MB

// Output sizes at which rows that are better whole begin to differ by more than the sample costs.
constexpr int64_t kManyBytes = int64_t{96} << 20, kMoreBytes = int64_t{256} << 20;
constexpr int64_t kVeryManyBytes = int64_t{1536} << 20;

// Which kinds of rows are computed whole, and by how many work-groups (us, by slices and whole):
// - Rows of one chunk (up to 512 channels in 16 bits) never: 400,000 rows over 100,000 of 512 in
//   bf16 274, 471, kept rows 114, 234; 100,000 over 50,000 of 128 (three quarters of the lanes idle
//   in whole rows) 17, 121.
// - Few rows never: their launch is short and the table's slices stay in the L2s.  bf16, 1,024
//   channels, kept rows: 32,928 over 16,464 21, 23.  Three chunks and more pass earlier: 60,000 over
//   20,000 of 1,536 55, 51 (184 MB), 24,576 over 12,288 of 1,024 in fp32 28, 25 (101 MB).  Below
//   that kept fp32 rows lose up to 2.4 us to the slices (16,447 over 8,231: 19.1, 16.7).
// - kKept: 1,048,576 over 65,536 of 1,024: bf16 590, 418; fp32 1,620, 984.
// - kOneHot where a table's slice is over three L2s: 262,144 over 262,144: bf16 262, 175; fp32 482,
//   355; 1,048,576 over 65,536 (8 MB) in bf16 633, 640.
// - kPart in 16 bits: bf16, 1,048,576 over 65,536: 1,039, 969, over 262,144: 1,188, 999; in fp16, whose
//   sums take fewer instructions, only past three L2s: 867, 938 and 1,126, 978.  fp32: 1,736, 1,852.
// - kNear in the largest calls, where the slices' waves drift apart: bf16 1,048,576 over 65,536: 1,017,
//   841, fp32 1,665, 1,431; but 205,800 over 52,968 203, 222 and 247, 372.
// - kMixed never: 1,238, 1,456 and 2,399, 2,932.
// A CU's whole rows want few waves, so that neighbours in flight share their parents' lines: 3
// work-groups where a row takes a wave four chunks (6 for the largest calls' kept rows, which share
// none), 5 for shorter rows.
template <typename T>
WholeRows whole_rule(const Rows<T>& r) {
  WholeRows whole;
  const int64_t out_bytes = r.out_bytes();
  const int64_t slice_bytes = r.table_rows * (sizeof(T) == 4 ? 256 : 128);
  const bool wide = r.chunks() >= 4;
  if (r.chunks() == 1 || out_bytes < (r.chunks() >= 3 ? kManyBytes : kMoreBytes)) return whole;
  const bool very_many = out_bytes >= kVeryManyBytes;
  const int cus = device_cus(), some = cus * (!wide ? 5 : very_many ? 6 : 3);
  whole.groups[kKept] = some;
  if (slice_bytes > (12 << 20)) whole.groups[kOneHot] = some;
  const bool slow_slices = std::is_same_v<T, bf16_t> || slice_bytes > (12 << 20);
  if (sizeof(T) == 2 && slow_slices && out_bytes >= 2 * kMoreBytes) whole.groups[kPart] = some;
  if (very_many && (wide || slow_slices))
    whole.groups[kNear] = cus * (wide ? 3 : 5);
  return whole;
}

template <typename T>
int launch_project(const void* table, int64_t table_stride, const int32_t* index,
                   const float* weight, const int32_t* order, void* out, int64_t out_stride,
                   int64_t n_rows, int64_t table_rows, int64_t dim, hipStream_t stream) {
  const Rows<T> r{static_cast<const T*>(table), table_stride, index, weight, order, static_cast<T*>(out), out_stride,
                  n_rows, table_rows, static_cast<int>(dim), stream};
  if (vector_rows<T>(table, table_stride, out, out_stride, dim)) {
    // Rows in an order have their repeats beside them (the figures at whole_rows), so they are
    // computed whole, but for 16-bit calls whose table the L2s hold anyway (32,928 rows over 16,464 of
    // 1,024 channels in bf16: 38 by slices, 53 whole; one-hot rows in fp16 24, 23).
    if (order != nullptr && r.chunks() >= 2 && (sizeof(T) == 4 || r.out_bytes() >= kManyBytes)) {
      launch_rows<T, false>(r, nullptr);
      return check_launch("top4_project");
    }
    const WholeRows whole = order == nullptr ? whole_rule(r) : WholeRows{};
    if constexpr (sizeof(T) == 4)
      launch_sliced<T, 16>(r, 4, whole);
    else if (table_rows <= kNarrowRows)
      launch_sliced<T, 8>(r, table_rows <= kHalfL2Rows ? 8 : 4, whole);
    else
      launch_sliced<T, 32>(r, 4, whole);
  } else {
    dim3 grid(static_cast<unsigned>((dim + 255) / 256), 1, 1);
    // Rows go on grid.y in slabs of 65535 (the y limit).
    for (int64_t r0 = 0; r0 < n_rows; r0 += 65535) {
      const int64_t nr = (n_rows - r0) < 65535 ? (n_rows - r0) : 65535;
      grid.y = static_cast<unsigned>(nr);
      hipLaunchKernelGGL((top4_project_scalar_kernel<T>), grid, dim3(256), 0, stream, r.table,
                         table_stride, index, weight, order, r.out, out_stride, n_rows, r0, table_rows,
                         r.dim);
    }
  }
  return check_launch("top4_project");
}

template <typename T>
int launch_probe(const void* table, int64_t table_stride, const int32_t* index, const float* weight,
                 int64_t n_rows, int64_t table_rows, int64_t dim, float* row_sums, hipStream_t stream) {
  if (!vector_rows<T>(table, table_stride, nullptr, dim, dim))
    return fail(VGO_EUNSUPPORTED, "top4_gather_probe: rows must be whole 16-byte chunks");
  launch_rows<T, true>({static_cast<const T*>(table), table_stride, index, weight, nullptr, nullptr, dim, n_rows,
                        table_rows, static_cast<int>(dim), stream}, row_sums);
  return check_launch("top4_gather_probe");
}

}  // namespace
}  // namespace vgo

namespace {
int project_entry(const void* table, int64_t table_row_stride, const int32_t* index,
                  const float* weight, const int32_t* order, void* out, int64_t out_row_stride,
                  int64_t n_rows, int64_t table_rows, int64_t dim, int dtype, void* stream) {
  using namespace vgo;
  VGO_REQUIRE(n_rows >= 0 && table_rows >= 0 && dim >= 0, "top4_project: negative size");
  if (n_rows == 0 || dim == 0) return VGO_OK;
  VGO_REQUIRE(index && weight && out, "top4_project: null pointer");
  VGO_REQUIRE(table || table_rows == 0, "top4_project: null table");
  VGO_REQUIRE(dim <= 0x7fffffff && n_rows <= 0x7fffffff, "top4_project: size too large");
  VGO_REQUIRE(table_row_stride >= dim && out_row_stride >= dim, "top4_project: row stride < dim");
  VGO_REQUIRE(aligned(index, 16) && aligned(weight, 16),
              "top4_project: index/weight must be 16-byte aligned [n,4] arrays");
  hipStream_t s = as_stream(stream);
  switch (dtype) {
    case VGO_F32:
      return launch_project<float>(table, table_row_stride, index, weight, order, out, out_row_stride,
                                   n_rows, table_rows, dim, s);
    case VGO_BF16:
      return launch_project<bf16_t>(table, table_row_stride, index, weight, order, out, out_row_stride,
                                    n_rows, table_rows, dim, s);
    case VGO_F16:
      return launch_project<f16_t>(table, table_row_stride, index, weight, order, out, out_row_stride,
                                   n_rows, table_rows, dim, s);
    default:
      return fail(VGO_EINVAL, "top4_project: unknown dtype");
  }
}
}  // namespace

extern "C" int vgo_top4_project(const void* table, int64_t table_row_stride, const int32_t* index,
                                const float* weight, void* out, int64_t out_row_stride,
                                int64_t n_rows, int64_t table_rows, int64_t dim, int dtype,
                                void* stream) {
  return project_entry(table, table_row_stride, index, weight, nullptr, out, out_row_stride, n_rows,
                       table_rows, dim, dtype, stream);
}

extern "C" int vgo_top4_gather_probe(const void* table, int64_t table_row_stride,
                                     const int32_t* index, const float* weight, float* row_sums,
                                     int64_t n_rows, int64_t table_rows, int64_t dim, int dtype,
                                     void* stream) {
  using namespace vgo;
  VGO_REQUIRE(n_rows >= 0 && table_rows >= 0 && dim >= 0, "top4_gather_probe: negative size");
  if (n_rows == 0 || dim == 0) return VGO_OK;
  VGO_REQUIRE(table && index && weight && row_sums, "top4_gather_probe: null pointer");
  VGO_REQUIRE(dim <= 0x7fffffff && n_rows <= 0x7fffffff && table_row_stride >= dim,
              "top4_gather_probe: bad size or stride");
  VGO_REQUIRE(aligned(index, 16) && aligned(weight, 16),
              "top4_gather_probe: index/weight must be 16-byte aligned [n,4] arrays");
  hipStream_t s = as_stream(stream);
  switch (dtype) {
    case VGO_F32:
      return launch_probe<float>(table, table_row_stride, index, weight, n_rows, table_rows, dim, row_sums, s);
    case VGO_BF16:
      return launch_probe<bf16_t>(table, table_row_stride, index, weight, n_rows, table_rows, dim, row_sums, s);
    case VGO_F16:
      return launch_probe<f16_t>(table, table_row_stride, index, weight, n_rows, table_rows, dim, row_sums, s);
    default:
      return fail(VGO_EINVAL, "top4_gather_probe: unknown dtype");
  }
}

extern "C" int vgo_top4_project_ordered(const void* table, int64_t table_row_stride,
                                        const int32_t* index, const float* weight,
                                        const int32_t* order, void* out, int64_t out_row_stride,
                                        int64_t n_rows, int64_t table_rows, int64_t dim, int dtype,
                                        void* stream) {
  using namespace vgo;
  VGO_REQUIRE(order || n_rows == 0, "top4_project_ordered: null order");
  return project_entry(table, table_row_stride, index, weight, order, out, out_row_stride, n_rows,
                       table_rows, dim, dtype, stream);
}
