// What the two sparse attention kernels (attn.hip, attn_few.hip) share.  Not
// part of the C ABI.
#pragma once

#include "sgl_common.h"
#include "sgl_rules.h"

namespace sgl {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef v4s __attribute__((address_space(3))) lds_v4s;

constexpr int kD = 512;     // head dim: 448 latent + 64 rope
constexpr int kBlk = 64;    // indices a split is cut by
constexpr int kHG = 64;     // heads per workgroup
constexpr int kARow = 584, kAData = 576, kANope = 448;
constexpr float kLog2e = 1.4426950408889634f;

struct AttnArgs {
  const uint16_t* q;   // [B, M, Hh, 512] bf16
  const uint8_t* kv;   // per batch element: bf16 [n, ld] | layout A [n, 584] | layout A pages
  int64_t n;           // rows per batch element
  int64_t kv_bstride;  // bytes between batch elements
  int64_t ld;          // bf16 rows: elements per row
  int page;            // footer pages: rows per page
  int page_shift;      // log2(page) when page is a power of two, else -1
  const float* sink;   // [Hh]
  const int32_t* idx;  // [B, M, K]
  int64_t M, K;
  int Hh;
  float scale;
  uint16_t* o;         // [B, M, Hh, 512] bf16
  int nsplit;          // > 1: the K rows are split over workgroups, partials to ws
  int bps;             // 64-row blocks per split
  float* ws_acc;       // [B, M, nsplit, Hh, 512] unnormalised outputs
  float* ws_ml;        // [B, M, nsplit, Hh, 2] running max (log2 units) and sum
};

// Row-major tile: token t, 16-byte chunk c (8 dims) at t*1024 + ((c ^ sw(t)) << 4).
// sw rotates the token's low four bits, which keeps conflict-free both the
// S^T fragment reads (16 B of one chunk from 16 consecutive tokens) and the
// transpose reads (8 B of 4 consecutive chunks from 4 consecutive tokens).
__device__ __forceinline__ uint32_t sw(int t) { return (uint32_t)(((t & 3) << 2) | ((t >> 2) & 3)); }

__device__ __forceinline__ v4s lds_tr16(const uint8_t* base, uint32_t off) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(base + off));
}

template <bool HI>
__device__ __forceinline__ uint32_t cvt2_e4m3_bf16(uint32_t w, float sc) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, sc, HI));
}

// attn_few.hip: at most 64 heads.
void launch_sparse_attn_few(const AttnArgs& a, int kv_format, dim3 grid, hipStream_t stream);

}  // namespace sgl
