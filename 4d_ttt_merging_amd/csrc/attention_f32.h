// fp32 mass-bias attention (attention_f32.hip), called by the C entries of attention.hip.
#pragma once

#include "vgo_common.h"

namespace vgo {

// One attention problem of a call, as the C ABI describes it.
struct Problem {
  const void* q;
  const void* k;
  const void* v;
  const void* bias;
  void* out;
  int64_t batch, heads, nq, nk;
  const int64_t* qs;
  const int64_t* ks;
  const int64_t* vs;
  const int64_t* os;
};

// Workspace bytes with which launch_attn_f32 may split tasks between work-groups.
size_t attn_f32_workspace(const Problem& p);
// With a workspace of at least attn_f32_workspace(p) bytes the key tiles are split evenly
// over the resident work-groups; with less (or none) every work-group runs whole tasks.
int launch_attn_f32(const Problem& p, void* workspace, size_t workspace_bytes, hipStream_t stream);

}  // namespace vgo
