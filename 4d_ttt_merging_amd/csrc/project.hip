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
#include <algorithm>

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
__global__ __launch_bounds__(kWaves * 64) void top4_project_kernel(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, const int32_t* __restrict__ order, T* __restrict__ out,
    int64_t out_stride, int64_t n_rows, int64_t table_rows, int dim, int n_slices) {
  typedef typename Vec16<T>::type V;
  constexpr int kGroup = 64 / W;
  constexpr int kRows = 2 * kGroup;
  const int lane = lane_id();
  const int xcd = blockIdx.x % kNumXcd;
  const int waves = static_cast<int>(gridDim.x) / kNumXcd * kWaves;  // of this XCD
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

// The gather probe (vgo_top4_gather_probe): whole-row gathers and the projection's
// arithmetic, but each row's output values are summed in fp32 (per lane, then over
// the wave) and only that sum is written, to row_sums[row]: what the fabric gives
// random whole-row reads.  Persistent waves, R consecutive rows gathered at once.
template <typename T, int R, int CH>
__global__ __launch_bounds__(kWaves * 64) void top4_gather_probe_kernel(
    const T* __restrict__ table, int64_t table_stride, const int32_t* __restrict__ index,
    const float* __restrict__ weight, int64_t n_rows, int64_t table_rows, int dim,
    float* __restrict__ row_sums) {
  typedef typename Vec16<T>::type V;
  constexpr int VN = Vec16<T>::n;
  const int lane = lane_id();
  const int64_t wave_gid = __builtin_amdgcn_readfirstlane(
      static_cast<int>(blockIdx.x) * kWaves + static_cast<int>(threadIdx.x >> 6));
  const int64_t step = static_cast<int64_t>(gridDim.x) * kWaves * R;
  for (int64_t r0 = wave_gid * R; r0 < n_rows; r0 += step) {
    Corners<T> corner[R];
    float lane_sum[R];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      corner[rr].load(index, weight, r0 + rr < n_rows ? r0 + rr : -1, table_rows);
      lane_sum[rr] = 0.0f;
    }
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
      for (int rr = 0; rr < R; ++rr)
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) {
          if (base + (ch * 64 + lane) * VN >= dim) continue;
          const V o = corner[rr].sum(y[rr][ch]);
#pragma unroll
          for (int j = 0; j < VN; ++j) lane_sum[rr] += to_f32(o[j]);
        }
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      float v = lane_sum[rr];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
      if (lane == 0 && r0 + rr < n_rows) row_sums[r0 + rr] = v;
    }
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

template <typename T, int W>
void launch_sliced(const T* tb, int64_t table_stride, const int32_t* index, const float* weight,
                   const int32_t* order, T* ob, int64_t out_stride, int64_t n_rows, int64_t table_rows,
                   int dim, int groups_per_cu, hipStream_t stream) {
  constexpr int kRows = 2 * 64 / W;
  const int n_slices = (dim + W * Vec16<T>::n - 1) / (W * Vec16<T>::n);
  const int64_t units = (n_rows + kRows - 1) / kRows * n_slices;
  const int64_t per_xcd = (units + kNumXcd - 1) / kNumXcd;
  const int64_t cap = std::max<int64_t>(1, int64_t{device_cus()} * groups_per_cu / kNumXcd);
  const int64_t groups = std::min<int64_t>(cap, (per_xcd + kWaves - 1) / kWaves);
  hipLaunchKernelGGL((top4_project_kernel<T, W>), dim3(static_cast<unsigned>(groups * kNumXcd)),
                     dim3(kWaves * 64), 0, stream, tb, table_stride, index, weight, order, ob,
                     out_stride, n_rows, table_rows, dim, n_slices);
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

template <typename T>
int launch_project(const void* table, int64_t table_stride, const int32_t* index,
                   const float* weight, const int32_t* order, void* out, int64_t out_stride,
                   int64_t n_rows, int64_t table_rows, int64_t dim, hipStream_t stream) {
  const T* tb = static_cast<const T*>(table);
  T* ob = static_cast<T*>(out);
  if (vector_rows<T>(table, table_stride, out, out_stride, dim)) {
    const int d = static_cast<int>(dim);
    if constexpr (sizeof(T) == 4) {
      launch_sliced<T, 16>(tb, table_stride, index, weight, order, ob, out_stride, n_rows, table_rows, d, 4, stream);
    } else if (table_rows <= kNarrowRows) {
      launch_sliced<T, 8>(tb, table_stride, index, weight, order, ob, out_stride, n_rows, table_rows, d,
                          table_rows <= kHalfL2Rows ? 8 : 4, stream);
    } else {
      launch_sliced<T, 32>(tb, table_stride, index, weight, order, ob, out_stride, n_rows, table_rows, d, 4, stream);
    }
  } else {
    dim3 grid(static_cast<unsigned>((dim + 255) / 256), 1, 1);
    // Rows go on grid.y in slabs of 65535 (the y limit).
    for (int64_t r0 = 0; r0 < n_rows; r0 += 65535) {
      const int64_t nr = (n_rows - r0) < 65535 ? (n_rows - r0) : 65535;
      grid.y = static_cast<unsigned>(nr);
      hipLaunchKernelGGL((top4_project_scalar_kernel<T>), grid, dim3(256), 0, stream, tb,
                         table_stride, index, weight, order, ob, out_stride, n_rows, r0, table_rows,
                         static_cast<int>(dim));
    }
  }
  return check_launch("top4_project");
}

template <typename T>
int launch_probe(const void* table, int64_t table_stride, const int32_t* index, const float* weight,
                 int64_t n_rows, int64_t table_rows, int64_t dim, float* row_sums, hipStream_t stream) {
  if (!vector_rows<T>(table, table_stride, nullptr, dim, dim))
    return fail(VGO_EUNSUPPORTED, "top4_gather_probe: rows must be whole 16-byte chunks");
  // 16-byte chunks per row per lane, and how many rows a wave gathers at once
  // (about 32 chunks = 512 B in flight per lane); eight work-groups per CU.
  const int row_chunks = static_cast<int>((dim + 64 * Vec16<T>::n - 1) / (64 * Vec16<T>::n));
  const int rows_per_wave = row_chunks >= 4 ? 2 : row_chunks >= 2 ? 4 : 8;
  const int64_t need = (n_rows + kWaves * rows_per_wave - 1) / (kWaves * rows_per_wave);
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>(need, int64_t{device_cus()} * 8)));
  const T* tb = static_cast<const T*>(table);
  const int d = static_cast<int>(dim);
  if (row_chunks >= 4)
    hipLaunchKernelGGL((top4_gather_probe_kernel<T, 2, 4>), grid, dim3(kWaves * 64), 0, stream, tb,
                       table_stride, index, weight, n_rows, table_rows, d, row_sums);
  else if (row_chunks >= 2)
    hipLaunchKernelGGL((top4_gather_probe_kernel<T, 4, 2>), grid, dim3(kWaves * 64), 0, stream, tb,
                       table_stride, index, weight, n_rows, table_rows, d, row_sums);
  else
    hipLaunchKernelGGL((top4_gather_probe_kernel<T, 8, 1>), grid, dim3(kWaves * 64), 0, stream, tb,
                       table_stride, index, weight, n_rows, table_rows, d, row_sums);
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
