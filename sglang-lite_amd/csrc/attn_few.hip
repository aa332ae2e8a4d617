// Sparse attention over a short chain of rows: few indices, or many splits, and
// at most 64 heads (the rule: attn_plan in sgl_rules.h; the semantics, and the
// kernel that does the rest: attn.hip).
//
// One workgroup per (query token, split of the rows).  Such a call is a chain
// of latencies: the indices, the rows, one to four blocks, the outputs.  So a
// block is 64 rows and goes through all steps before the next one, which saves
// the phases that attn.hip runs ahead to fill its waits (worth it from three
// or four blocks, sooner with more heads): one query x 8 heads x 64 indices of
// packed pages 7.6 us where attn.hip takes 10.0, x 256 10.8 and 13.5.  Valid rows
// are not packed; blocks at the end with every entry masked are left out (2048
// queries x 8 heads x 192 indices, bf16, 30 % valid: 89.8 us with them, 54.3
// without, attn.hip 64.0).
// Eight wavefronts; per block:
//   gather:  each wavefront dequantizes 8 rows (loaded during the previous
//            block) into one row-major bf16 tile in LDS (swizzled);
//   S^T = KV . Q^T (v_mfma_f32_32x32x16_bf16, Q^T fragments parked in LDS):
//            of 32 heads, wavefront dq = 2 dh + th the partial of the 32 tokens
//            of half th over dims [256 dh, +256); the partials meet in LDS and
//            each of the heads' four wavefronts sums and finishes the softmax
//            (identically);
//   O^T += V^T . P^T: P^T is the S^T accumulator itself, cast to bf16 (the
//            32x32 output layout of S^T is the B operand layout of the next
//            MFMA), and V^T fragments come straight from the row-major tile
//            with ds_read_b64_tr_b16; each wavefront its 128 dims.
// In both products lane (head c, half g) owns head c: the running max, sum
// and rescale factor of a head live in the lanes that hold its outputs.  At
// most 32 heads keep wavefronts 0-3 busy, one per SIMD (with two on each of
// two SIMDs one query x 8 heads x 64 indices took 8.5 us).
#include "sgl_attn.h"
#include "sgl_numeric.h"

namespace sgl {
namespace {

typedef short v8s __attribute__((ext_vector_type(8)));

// HG: 32-head groups of the workgroup (1: at most 32 heads, 2: at most 64).
template <int FMT, int HG>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sparse_attn_few_kernel(const AttnArgs a) {
  __shared__ __align__(16) uint8_t sKV[kBlk * 1024];
  __shared__ __align__(16) uint4 sQ[HG][2][16][64];    // Q^T fragments, [hg][dh][ks][lane]
  __shared__ __align__(16) float4 sS[HG][4][4][64];    // S^T partials, [hg][dq][quad][lane]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // wavefront (hg, dq): heads [32 hg, +32); S^T over dims [256 dh, +256) for
  // tokens [32 th, +32) of a block (dq = 2 dh + th), and O^T over dims
  // [128 dq, +128) for all 64 tokens (HG = 1: wavefronts 4-7 gather only)
  const int hg = HG == 1 ? wave >> 2 : wave & 1, dq = HG == 1 ? wave & 3 : wave >> 1;
  const int dh = dq >> 1, th = dq & 1;
  const int h0 = 32 * hg;
  const bool active = hg < HG;
  const int g2 = lane >> 5, c32 = lane & 31;
  const int64_t m = attn_query_in_seq(blockIdx.x, (uint32_t)a.M), b = blockIdx.y;
  const int split = (int)blockIdx.z;
  const uint8_t* kvb = a.kv + b * a.kv_bstride;
  const int32_t* idxp = a.idx + (b * a.M + m) * a.K;

  // S^T A operand: token 32 th + c32, chunk 32 dh + 2 ks + g2; the swizzle
  // only touches the chunk's low four bits, so ks % 8 picks one of eight
  // bases and the rest is an immediate offset
  uint32_t qa[8];
#pragma unroll
  for (int k8 = 0; k8 < 8; ++k8)
    qa[k8] = (32 * th + c32) * 1024 + 512 * dh + ((((2 * k8 + g2) ^ sw(c32)) & 15) << 4);
  // V^T A operand by transpose read: in each 16-lane group G, source lane s
  // reads 4 dims of token 16 s4 + 8 e + 4 (G >> 1) + (s >> 2), and the read
  // hands each lane 4 consecutive tokens of one dim, i.e. 4 consecutive K
  // elements of one row of V^T.  Bases for each (e, dt).
  uint32_t va[2][4];
  {
    const int G = lane >> 4, s16 = lane & 15;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const int tok = 8 * e + 4 * (G >> 1) + (s16 >> 2);
        const int cl = 4 * dt + 2 * (G & 1) + ((s16 & 3) >> 1);
        va[e][dt] = tok * 1024 + 256 * dq + ((cl ^ sw(tok)) << 4) + 8 * (s16 & 1);
      }
  }

  v16f acc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.0f;
  const float NEG_INF = -__builtin_huge_valf();
  const float c1 = a.scale * kLog2e;
  float m_run = NEG_INF, l_run = 0.0f;  // head c32: reference point (log2 units) and sum

  // layout A per-lane byte offsets: lanes < 56 take 8 e4m3 bytes and the
  // row's 8-byte scale footer, lanes 56..63 the 16 rope bytes in two halves
  const bool nope_lane = lane < 56;
  const uint32_t o0 = nope_lane ? 8 * lane : kANope + 16 * (lane - 56);
  const uint32_t o1r = kANope + 8 + 16 * (lane - 56);  // rope second half (rope lanes)
  const int sb_shift = 8 * ((lane >> 3) & 3);
  const bool sb_hi = (lane >> 3) >= 4;

  // A block's indices are loaded unconditionally (clamped to the last one)
  // and checked where they are used: the check waits for the load, and since
  // loads complete in order, a check right after the load would also wait
  // for every row gather issued before it.
  auto load_ids = [&](int j) -> int32_t {
    const int64_t p = (int64_t)j * kBlk + lane;
    return idxp[p < a.K ? p : a.K - 1];
  };
  auto check_id = [&](int j, int32_t id) -> int32_t {
    const int64_t p = (int64_t)j * kBlk + lane;
    return (p < a.K && id >= 0 && id < a.n) ? id : -1;
  };
  // this wavefront's 8 rows of the block: tokens 8 wave + rr.  The gathers
  // are unconditional (a missing row reads row 0, which store_rows zeroes),
  // so no branch splits the loads and the compiler's wait before the stores
  // counts the loads in flight instead of draining them.
  uint4 raw[8];
  auto load_rows = [&](int32_t ids) {
    if (a.n == 0) return;  // no rows at all: store_rows zeroes every row
#pragma unroll
    for (int rr = 0; rr < 8; ++rr) {
      const int idr = __builtin_amdgcn_readlane(ids, 8 * wave + rr);
      const int id = idr >= 0 ? idr : 0;
      uint4 v;
      {
        if constexpr (FMT == SGL_ATTN_KV_BF16) {
          v = *reinterpret_cast<const uint4*>(kvb + (int64_t)id * a.ld * 2 + lane * 16);
        } else {
          const uint8_t* data;
          const uint8_t* foot;
          if constexpr (FMT == SGL_ATTN_KV_A_PAGED) {
            const int pg = a.page_shift >= 0 ? id >> a.page_shift : (int)((uint32_t)id / (uint32_t)a.page);
            const int l = id - pg * a.page;
            const uint8_t* pbase = kvb + (int64_t)pg * a.page * kARow;
            data = pbase + l * kAData;
            foot = pbase + a.page * kAData + l * 8;
          } else {
            data = kvb + (int64_t)id * kARow;
            foot = data + kAData;
          }
          const uint2 x = *reinterpret_cast<const uint2*>(data + o0);
          const uint2 y = *reinterpret_cast<const uint2*>(nope_lane ? foot : data + o1r);
          v = make_uint4(x.x, x.y, y.x, y.y);
        }
      }
      raw[rr] = v;
    }
  };
  auto store_rows = [&](int32_t ids) {
#pragma unroll
    for (int rr = 0; rr < 8; ++rr) {
      uint4 v = raw[rr];
      if (__builtin_amdgcn_readlane(ids, 8 * wave + rr) < 0) v = make_uint4(0, 0, 0, 0);
      if constexpr (FMT != SGL_ATTN_KV_BF16) {
        const uint32_t word = sb_hi ? v.w : v.z;
        const float sc = bits_f32(((word >> sb_shift) & 0xFFu) << 23);  // 2^(e8m0 - 127)
        // word by word: a select of whole uint4 values goes through scratch
        const uint32_t c0 = cvt2_e4m3_bf16<false>(v.x, sc), c1 = cvt2_e4m3_bf16<true>(v.x, sc);
        const uint32_t c2 = cvt2_e4m3_bf16<false>(v.y, sc), c3 = cvt2_e4m3_bf16<true>(v.y, sc);
        v.x = nope_lane ? c0 : v.x;
        v.y = nope_lane ? c1 : v.y;
        v.z = nope_lane ? c2 : v.z;
        v.w = nope_lane ? c3 : v.w;
      }
      const int t = 8 * wave + rr;
      *reinterpret_cast<uint4*>(sKV + t * 1024 + ((lane ^ sw(t)) << 4)) = v;
    }
  };

  const int nblk_all = (int)((a.K + kBlk - 1) / kBlk);
  const int jb = split * a.bps;  // this split's first block
  int nblk = jb + a.bps < nblk_all ? jb + a.bps : nblk_all;
  // indices run two blocks ahead of the MFMAs, the rows one block ahead;
  // past the last block the loads repeat it (their results are unused)
  int32_t ids = jb < nblk ? load_ids(jb) : -1;
  // blocks at the end with every entry masked are left out (not those between
  // others: a branch in the loop would split its loads)
  while (nblk > jb + 1 && __ballot(check_id(nblk - 1, load_ids(nblk - 1)) >= 0) == 0) --nblk;
  ids = check_id(jb, ids);
  int32_t ids_next = jb < nblk ? load_ids(jb + 1 < nblk ? jb + 1 : jb) : -1;  // raw (none when K == 0)
  load_rows(ids);
  // Q^T B operand: lane (head c32, half g2) of step ks holds
  // q[h0 + c32][256 dh + 16 ks + 8 g2, +8); the two token halves share it.
  // Loaded after the first rows' gathers are issued, so its memory latency
  // overlaps theirs: the first block waits for two memory round trips (the
  // indices, then the rows with Q), not three
  if (active) {
    const int h = min(h0 + c32, a.Hh - 1);
    const uint16_t* qrow = a.q + ((b * a.M + m) * a.Hh + h) * (int64_t)kD + 256 * dh + 8 * g2;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int ks = 8 * th + k;
      sQ[hg][dh][ks][lane] = *reinterpret_cast<const uint4*>(qrow + 16 * ks);
    }
  }
  for (int j = jb; j < nblk; ++j) {
    const uint64_t valid = __ballot(ids >= 0);
    __syncthreads();  // the previous block's tile is consumed
    store_rows(ids);
    __syncthreads();  // block j (and, the first time, Q) is in LDS
    {
      const int jn = j + 1 < nblk ? j + 1 : j;
      ids = j + 1 < nblk ? check_id(jn, ids_next) : -1;
      ids_next = load_ids(j + 2 < nblk ? j + 2 : jn);  // before the rows it would wait behind
      load_rows(ids);
    }
    if (!active) {
      __syncthreads();  // (partials exchanged)
      continue;
    }
    // partial S^T of tile th over dims [256 dh, +256): lane (head c32, g2)
    // gets token 32 th + 8 (r / 4) + 4 g2 + r % 4 in sp[r]
    v16f sp;
#pragma unroll
    for (int r = 0; r < 16; ++r) sp[r] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
      const v8bf qf = __builtin_bit_cast(v8bf, sQ[hg][dh][ks][lane]);
      const v8bf kvf = *reinterpret_cast<const v8bf*>(sKV + qa[ks & 7] + 256 * (ks >> 3));
      sp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kvf, qf, sp, 0, 0, 0);
    }
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      sS[hg][dq][q4][lane] = make_float4(sp[4 * q4], sp[4 * q4 + 1], sp[4 * q4 + 2], sp[4 * q4 + 3]);
    __syncthreads();  // partials exchanged
    // full S^T of both tiles: tile tt = partial (dh 0) + partial (dh 1), the
    // same sum in each of the four wavefronts
    v16f s[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      // (dh = 0 / 1, th = tt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const float4 x = sS[hg][tt][q4][lane], y = sS[hg][2 + tt][q4][lane];
        s[tt][4 * q4] = x.x + y.x;
        s[tt][4 * q4 + 1] = x.y + y.y;
        s[tt][4 * q4 + 2] = x.z + y.z;
        s[tt][4 * q4 + 3] = x.w + y.w;
      }
    }
    if (valid != ~0ull) {
      const uint64_t vl = g2 ? (valid >> 4) : valid;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (!((vl >> (32 * tt + 8 * (r >> 2) + (r & 3))) & 1ull)) s[tt][r] = NEG_INF;
    }
    // online softmax of head c32 (scale > 0: max(s) * c1 = max(s * c1))
    float mx = NEG_INF;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = __builtin_fmaxf(mx, s[tt][r]);
    mx = __builtin_fmaxf(mx, __shfl_xor(mx, 32, 64));
    // The reference point moves only when the block maximum exceeds it by
    // more than 8 (log2 units): the probabilities stay <= 256 (exact range
    // in bf16, same relative rounding) and the accumulator is rarely
    // rescaled.  Any reference >= the running max gives the same softmax.
    const float m_blk = mx * c1;
    const bool move = !(m_blk <= m_run + 8.0f);  // also true while m_run = -inf
    const float m_new = move ? __builtin_fmaxf(m_run, m_blk) : m_run;
    const float ref = m_new == NEG_INF ? 0.0f : m_new;  // a fully masked prefix keeps o = 0
    const float alpha = move ? __builtin_amdgcn_exp2f(m_run - ref) : 1.0f;
    float ls = 0.0f;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[tt][r], c1, -ref));
        ls += p;
        s[tt][r] = p;
      }
    ls += __shfl_xor(ls, 32, 64);
    l_run = l_run * alpha + ls;
    m_run = m_new;
    // P^T B operands: K step s4 (16 tokens) = tile s4 / 2, registers 8 (s4 % 2) + e
    v8bf pb[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      v8s w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t pk = pk2_bf16(s[s4 >> 1][8 * (s4 & 1) + 2 * e], s[s4 >> 1][8 * (s4 & 1) + 2 * e + 1]);
        w[2 * e] = (short)(pk & 0xFFFFu);
        w[2 * e + 1] = (short)(pk >> 16);
      }
      pb[s4] = __builtin_bit_cast(v8bf, w);
    }
    if (j > jb && __ballot(alpha != 1.0f)) {  // (the accumulator is zero before the first block)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] *= alpha;
    }
    // O^T += V^T . P^T over this wavefront's 4 tiles of 32 dims (K step
    // outer: four independent accumulators between dependent MFMAs)
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const v4s lo = lds_tr16(sKV, va[0][dt] + 16384 * s4);
        const v4s hi = lds_tr16(sKV, va[1][dt] + 16384 * s4);
        const v8bf vf = __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pb[s4], acc[dt], 0, 0, 0);
      }
    }
  }
  const int h = h0 + c32;
  if (!active || h >= a.Hh) return;
  // lane (head h, g2) holds dims 128 dq + 32 dt + 8 (r / 4) + 4 g2 + r % 4 in acc[dt][r]
  if (a.nsplit > 1) {
    const int64_t qs = (b * a.M + m) * a.nsplit + split;
    if (dq == 0 && g2 == 0) {
      float* ml = a.ws_ml + (qs * a.Hh + h) * 2;
      ml[0] = m_run;
      ml[1] = l_run;
    }
    float* row = a.ws_acc + (qs * a.Hh + h) * (int64_t)kD + 128 * dq + 4 * g2;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *reinterpret_cast<float4*>(row + 32 * dt + 8 * q4) =
            make_float4(acc[dt][4 * q4], acc[dt][4 * q4 + 1], acc[dt][4 * q4 + 2], acc[dt][4 * q4 + 3]);
    return;
  }
  // o = acc / (l + exp(sink - m))
  const float ref = m_run == NEG_INF ? 0.0f : m_run;
  const float inv = 1.0f / (l_run + __builtin_amdgcn_exp2f(a.sink[h] * kLog2e - ref));
  uint16_t* orow = a.o + ((b * a.M + m) * a.Hh + h) * (int64_t)kD + 128 * dq + 4 * g2;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      *reinterpret_cast<uint2*>(orow + 32 * dt + 8 * q4) =
          make_uint2(pk2_bf16(acc[dt][4 * q4] * inv, acc[dt][4 * q4 + 1] * inv),
                     pk2_bf16(acc[dt][4 * q4 + 2] * inv, acc[dt][4 * q4 + 3] * inv));
}

}  // namespace

void launch_sparse_attn_few(const AttnArgs& a, int kv_format, dim3 grid, hipStream_t st) {
#define SGL_ATTN_FEW(FMT)                                              \
  do {                                                                 \
    if (a.Hh <= 32)                                                    \
      sparse_attn_few_kernel<FMT, 1><<<grid, 512, 0, st>>>(a);         \
    else                                                               \
      sparse_attn_few_kernel<FMT, 2><<<grid, 512, 0, st>>>(a);         \
  } while (0)
  if (kv_format == SGL_ATTN_KV_BF16)
    SGL_ATTN_FEW(SGL_ATTN_KV_BF16);
  else if (kv_format == SGL_ATTN_KV_A)
    SGL_ATTN_FEW(SGL_ATTN_KV_A);
  else
    SGL_ATTN_FEW(SGL_ATTN_KV_A_PAGED);
#undef SGL_ATTN_FEW
}

}  // namespace sgl
