// Exact (erf) GELU of bf16 values: out = x * 0.5 * (1 + erf(x / sqrt 2)) in fp32 with one
// rounding, the MLP activation of vggt_omega/models/layers/mlp.py under bf16 autocast.
//
// Bound: HBM.  Evaluated per element, erf takes longer than the 4 bytes of traffic:
// torch's kernel runs 32,928 x 4,096 values (540 MB) in 122 us; this one in 107, a
// copy of the same rows in 100 (5.4 TB/s).
// A bf16 value has few forms, so each work-group first evaluates the function for
// every value it is not trivial at (2^-14 <= |x| < 8: 2 x 2,176 values, 8.5 KB of LDS,
// four or five per lane) and then looks elements up, five instructions and one 2-byte
// LDS read each.  Below that range erf cannot move the rounding of x / 2, above
// it the fp32 erf is +-1; a wave with such an element takes the direct products.
// One 16-wave work-group per CU: the table is built once per CU.
#include <algorithm>

#include "vgo_common.h"

namespace vgo {
namespace {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 1024;
constexpr unsigned kLow = (127 - 14) << 7;           // bf16 bits of 2^-14
constexpr unsigned kValues = ((127 + 3) << 7) - kLow;  // up to 8, exclusive
static_assert(4 * kValues < 65536, "byte offsets of the table fit 16 bits");

__device__ __forceinline__ float value_of(unsigned bits) { return __builtin_bit_cast(float, bits << 16); }
__device__ __forceinline__ unsigned bits_of(float x) {
  return __builtin_bit_cast(unsigned short, from_f32<bf16_t>(x));
}

// An element in or out of the table's range.
__device__ __forceinline__ unsigned lookup_any(const unsigned short* table, unsigned bits) {
  const unsigned mag = bits & 0x7fffu, sign = bits >> 15;
  if (mag - kLow < kValues) return table[mag - kLow + sign * kValues];
  return bits_of(value_of(bits) * 0.5f * (mag < kLow ? 1.0f : sign ? 0.0f : 2.0f));
}

__device__ __forceinline__ u32x4 gelu8(const unsigned short* table, u32x4 x) {
  u16x2 u[4], last = {0, 0};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned word = x[i];  // a cast of the vector's element itself takes element 0
    const u16x2 b = __builtin_bit_cast(u16x2, word);
    u[i] = (b & static_cast<unsigned short>(0x7fff)) - static_cast<unsigned short>(kLow);  // wraps below the range
    last = __builtin_elementwise_max(last, u[i]);
    u[i] = u[i] + (b >> static_cast<unsigned short>(15)) * static_cast<unsigned short>(kValues);
  }
  u32x4 y;
  if (__builtin_expect(__any(max(last[0], last[1]) >= kValues), 0)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = lookup_any(table, x[i] & 0xffffu) | lookup_any(table, x[i] >> 16) << 16;
    return y;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    y[i] = static_cast<unsigned>(table[u[i][0]]) | static_cast<unsigned>(table[u[i][1]]) << 16;
  return y;
}

// x and out may be the same rows: every lane reads its 16 bytes before it writes them.
__global__ __launch_bounds__(kThreads, 4) void gelu_kernel(const bf16_t* x, bf16_t* out, int64_t n) {
  __shared__ unsigned short table[2 * kValues];
  for (unsigned i = threadIdx.x; i < 2 * kValues; i += kThreads) {
    const float v = value_of(i < kValues ? kLow + i : 0x8000u + kLow + i - kValues);
    table[i] = static_cast<unsigned short>(bits_of(v * 0.5f * (1.0f + erff(v * 0.70710678118654752440f))));
  }
  __syncthreads();
  const int64_t vectors = n / 8, step = static_cast<int64_t>(gridDim.x) * kThreads;
  const u32x4* src = reinterpret_cast<const u32x4*>(x);
  u32x4* dst = reinterpret_cast<u32x4*>(out);
  int64_t v = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  for (; v + 3 * step < vectors; v += 4 * step) {  // four vectors in flight per lane
    u32x4 a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = src[v + i * step];
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[v + i * step] = gelu8(table, a[i]);
  }
  for (; v < vectors; v += step) dst[v] = gelu8(table, src[v]);
  const int64_t tail = vectors * 8 + threadIdx.x;
  if (blockIdx.x == 0 && tail < n)
    reinterpret_cast<unsigned short*>(out)[tail] = static_cast<unsigned short>(
        lookup_any(table, reinterpret_cast<const unsigned short*>(x)[tail]));
}

}  // namespace
}  // namespace vgo

extern "C" int vgo_gelu_bf16(const void* x, void* out, int64_t n, void* stream) {
  using namespace vgo;
  VGO_REQUIRE(n >= 0, "gelu: negative size");
  if (n == 0) return VGO_OK;
  VGO_REQUIRE(x && out, "gelu: null pointer");
  VGO_REQUIRE(aligned(x, 16) && aligned(out, 16), "gelu: values must be 16-byte aligned");
  const int64_t groups = std::min<int64_t>(device_cus(), (n / 8 + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(gelu_kernel, dim3(static_cast<unsigned>(std::max<int64_t>(1, groups))), dim3(kThreads), 0,
                     as_stream(stream), static_cast<const bf16_t*>(x), static_cast<bf16_t*>(out), n);
  return check_launch("gelu");
}
