// Internal interface of the K-group dense FP8 GEMM (dense_mid.hip).  Not part
// of the C ABI.
#pragma once

#include "sgl_gemm.h"

namespace sgl {

constexpr int kNoMid = 1;
// The product on tiles that give at most one workgroup per CU, or kNoMid when
// there is no such tile; else the launch status.
int launch_dense_mid(GemmArgs& a, hipStream_t stream);

}  // namespace sgl
