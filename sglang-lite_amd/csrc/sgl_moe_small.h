// Internal interface of the smallest batches' expert layer (moe_small.hip).
// Not part of the C ABI.
#pragma once

#include "sgl_common.h"
#include "sgl_rules.h"

namespace sgl {

struct SmallMoeArgs {
  const uint8_t* xq;  // [T, H] e4m3
  const float* xs;    // [T, H/128]
  const int32_t* ids;
  const float* route_w;
  const sgl_expert_ptrs* experts;
  int64_t T, H, I;
  int E, k, has_shared;
  float swiglu_limit;
  int scale_mode;
  int sa_pow2;   // activation scales (x's and h's) are powers of two
  uint16_t* h;   // bf16 [T (k + has_shared), I]: slot rows, then the shared expert's
  uint16_t* y;   // bf16 [T, H]
};

// (the sizes: small_moe_ok)
int launch_small_moe(const SmallMoeArgs& args, bool fp4, hipStream_t stream);

}  // namespace sgl
