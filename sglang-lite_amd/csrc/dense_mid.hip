// Dense block-scaled FP8 GEMM for middling M: tiles of one workgroup per CU
// whose wavefronts split K between them.
//
// C[M, N] = sum_kb (A[:, kb] . B[:, kb]^T) sa[m, kb] sb[n/128, kb], as
// gemm_fp8_kernel computes it.  What bounds those tiles at M = 65 ... 512 is
// neither memory (M = 200, N = 4096, K = 7168: 84 % of their reads hit L2) nor
// the matrix cores (busy 9 % of the time) but the serial chain of a 128-deep stage (wait, barrier, fragment reads,
// MFMAs, promotion, the next loads' issue: about 1070 cycles at one workgroup
// of four wavefronts a CU), 56 times over at K = 7168.  So here a stage holds
// G K blocks, each computed by four wavefronts of its own over the whole tile,
// and the chain is walked K / (128 G) times; the G partial tiles are summed in
// order through LDS at the end.  Every K block's scales are staged in LDS
// first, so the loop's only memory instructions are the operand DMAs (whole
// 128-byte lines, the swizzle of the other kernels, NS - 1 stages ahead).
//
// N = 4096, K = 7168, e8m0 scales, graph-replayed over cold weights, the tiles
// before (32 x 64 ... 64 x 128, one K block a stage) / these: M = 128 19.1 / 12.2
// us (the weight alone reads in 7), 200 26.5 / 18.8, 512 40.0 / 26.1; N = 512:
// M = 512 39.1 / 12.0; K = 2048, N = 4096: M = 128 8.2 / 6.3, 512 15.4 / 10.6; fp32
// scales, M = 128 / 200 / 512 21.4 / 13.1, 28.3 / 23.2 (by the trace) and 35.2 / 30.0.
#include "sgl_gemm.h"
#include "sgl_dense_mid.h"
#include "sgl_numeric.h"

namespace sgl {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <int BM_, int BN_, int G_, int NS_, int MAXKB_>
struct MidCfg {
  static constexpr int BM = BM_, BN = BN_, G = G_, NS = NS_, MAXKB = MAXKB_;
  static constexpr int NW = 4 * G;                  // wavefronts: four (side by side along N) per K block
  static constexpr int TM = BM / 16, TN = BN / 64;  // 16 x 16 tiles of a wavefront
  static constexpr int BLK = (BM + BN) * 128;       // operand bytes of a K block
  static constexpr int STAGE = G * BLK;
  static constexpr int DPW = (BM + BN) / 8 / 4;     // 1 KB DMAs of a wavefront per stage
  static constexpr int LDS = NS * STAGE + MAXKB * BM * 4 + MAXKB * 4;
  static_assert((BM + BN) / 8 % 4 == 0 && BM / 8 % 4 == 0, "a wavefront's DMAs: A's first, then B's");
  static_assert(G * BM * BN * 4 <= NS * STAGE, "the partial tiles fit the ring");
  static_assert(LDS <= 160 * 1024, "the LDS of a CU");
};

// SCALED: both scales e8m0, applied inside the MFMA; else promoted in fp32.
template <class C, bool SCALED>
__global__ __launch_bounds__(64 * C::NW) void gemm_mid_kernel(const GemmArgs args) {
  constexpr int BM = C::BM, BN = C::BN, G = C::G, NS = C::NS, TM = C::TM, TN = C::TN;
  __shared__ __align__(16) uint8_t ring[NS * C::STAGE];
  __shared__ __align__(16) float sSa[C::MAXKB][BM];  // [K block][row]: fp32, or the e8m0 byte (SCALED)
  __shared__ float sSb[C::MAXKB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave >> 2, wn = wave & 3;  // K block of a stage, columns [wn BN / 4, + BN / 4)
  const int g4 = lane >> 4, r16 = lane & 15;
  const int64_t M = args.M, N = args.N, K = args.K;
  const int KB = (int)(K / 128), NST = (KB + G - 1) / G;

  // a contiguous range of tiles per XCD, M tiles of one weight slice adjacent
  const int mt = (int)((M + BM - 1) / BM), total = mt * args.n_tiles;
  const int per = (total + 7) >> 3, L = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || L >= total) return;
  const int nt = L / mt;
  const int64_t m0 = (int64_t)(L - nt * mt) * BM, n0 = (int64_t)nt * BN;

  // ---- this wavefront's DMAs of a stage: 8 rows x 128 bytes of its K block,
  // chunks wn + 4 j of [A rows | B rows]; rows past the end re-read the last
  uint64_t src[C::DPW];
  {
    const int rr = lane >> 3, pc = lane & 7;
#pragma unroll
    for (int j = 0; j < C::DPW; ++j) {
      const int c = wn + 4 * j, row = 8 * c + rr;  // row of [A | B]
      const bool isa = j < BM / 32;
      int64_t r = isa ? m0 + row : n0 + row - BM;
      const int64_t last = (isa ? M : N) - 1;
      if (r > last) r = last;
      src[j] = (uint64_t)(uintptr_t)(isa ? args.a : args.b) + (uint64_t)(r * K) + (uint64_t)((pc ^ swz(row)) << 4);
    }
  }
  const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_u32(ring));
  auto issue = [&](int st) {
    const int kb = st * G + g;
    if (kb >= KB) return;
    const uint32_t dst = ring_lds + (uint32_t)((st % NS) * C::STAGE + g * C::BLK);
#pragma unroll
    for (int j = 0; j < C::DPW; ++j) dma16v(src[j] + (uint64_t)kb * 128, dst + (uint32_t)((wn + 4 * j) * 1024));
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < NST) issue(s);

  // ---- scales
  for (int i = tid; i < BM * KB; i += 64 * C::NW) {
    const int r = i / KB, kb = i - r * KB;
    const int64_t row = m0 + r < M ? m0 + r : M - 1;
    float v;
    if (args.sa_e8m0) {
      const uint32_t b = reinterpret_cast<const uint8_t*>(args.sa)[row * KB + kb];
      v = SCALED ? bits_f32(b) : (b == 0xFFu ? bits_f32(0x7FC00000u) : (b == 0 ? bits_f32(0x00400000u) : bits_f32(b << 23)));
    } else {
      v = reinterpret_cast<const float*>(args.sa)[row * KB + kb];
    }
    sSa[kb][r] = v;
  }
  for (int kb = tid; kb < KB; kb += 64 * C::NW) {
    float v;
    if (args.sb_e8m0) {
      const uint32_t b = reinterpret_cast<const uint8_t*>(args.sb)[(n0 / 128) * KB + kb];
      v = SCALED ? bits_f32(b) : (b == 0xFFu ? bits_f32(0x7FC00000u) : (b == 0 ? bits_f32(0x00400000u) : bits_f32(b << 23)));
    } else {
      v = reinterpret_cast<const float*>(args.sb)[(n0 / 128) * KB + kb];
    }
    sSb[kb] = v;
  }

  const int c0 = ((2 * g4) ^ swz(r16)) << 4, c1 = ((2 * g4 + 1) ^ swz(r16)) << 4;
  auto frag = [&](const uint8_t* base) -> v8i {
    const uint4 lo = *reinterpret_cast<const uint4*>(base + r16 * 128 + c0);
    const uint4 hi = *reinterpret_cast<const uint4*>(base + r16 * 128 + c1);
    return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };
  v4f acc[TM][TN];
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero;

  for (int st = 0; st < NST; ++st) {
    // stage st landed (the younger stages' DMAs may be in flight; a wavefront
    // whose last K block does not exist has fewer), everyone done with st - 1
    if (NS > 2 && st + NS - 1 < NST)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NS - 2) * C::DPW) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (st + NS - 1 < NST) issue(st + NS - 1);
    const int kb = st * G + g;
    if (kb < KB) {
      const uint8_t* tA = ring + (st % NS) * C::STAGE + g * C::BLK;
      const uint8_t* tB = tA + (BM + wn * (BN / 4)) * 128;
      v8i bf[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = frag(tB + j * 2048);
      const float sb = sSb[kb];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const v8i af = frag(tA + i * 2048);
        if constexpr (SCALED) {
          const int sa = (int)f32_bits(sSa[kb][16 * i + r16]);
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[j], acc[i][j], 0, 0, 0, sa, 0,
                                                                        (int)f32_bits(sb));
        } else {
          const float4 sa = *reinterpret_cast<const float4*>(&sSa[kb][16 * i + 4 * g4]);
          const float s4[4] = {sa.x * sb, sa.y * sb, sa.z * sb, sa.w * sb};
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf[j], zero, 0, 0, 0, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(p[r], s4[r], acc[i][j][r]);
          }
        }
      }
    }
  }

  // ---- the G partial tiles through LDS (row-major, 16 columns' shift per
  // four rows so the lanes' writes spread over the banks), summed in order
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float* part = reinterpret_cast<float*>(ring);
  auto at = [&](int row, int col) -> int { return row * BN + ((col + 16 * (row >> 2)) & (BN - 1)); };
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[g * BM * BN + at(16 * i + 4 * g4 + r, wn * (BN / 4) + 16 * j + r16)] = acc[i][j][r];
  __syncthreads();
  for (int i = tid; i < BM * BN / 8; i += 64 * C::NW) {
    const int row = i / (BN / 8), col = (i - row * (BN / 8)) * 8;
    if (m0 + row >= M || n0 + col >= N) continue;
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; u += 4) {
      const float4 p = *reinterpret_cast<const float4*>(part + at(row, col + u));
      v[u] = p.x; v[u + 1] = p.y; v[u + 2] = p.z; v[u + 3] = p.w;
    }
#pragma unroll
    for (int q = 1; q < G; ++q)
#pragma unroll
      for (int u = 0; u < 8; u += 4) {
        const float4 p = *reinterpret_cast<const float4*>(part + q * BM * BN + at(row, col + u));
        v[u] += p.x; v[u + 1] += p.y; v[u + 2] += p.z; v[u + 3] += p.w;
      }
    const int64_t o = (m0 + row) * N + n0 + col;  // (N % 16 == 0: a group of 8 columns is whole)
    if (args.out_f32) {
      float4* c = reinterpret_cast<float4*>(reinterpret_cast<float*>(args.c) + o);
      c[0] = make_float4(v[0], v[1], v[2], v[3]);
      c[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(args.c) + o) =
          make_uint4(pk2_bf16_exact(v[0], v[1]), pk2_bf16_exact(v[2], v[3]), pk2_bf16_exact(v[4], v[5]),
                     pk2_bf16_exact(v[6], v[7]));
    }
  }
}

template <class C>
int launch_mid(GemmArgs& a, hipStream_t st) {
  a.n_tiles = (int)ceil_div(a.N, (int64_t)C::BN);
  const int64_t total = ceil_div(a.M, (int64_t)C::BM) * a.n_tiles;
  const unsigned grid = (unsigned)(8 * ((total + 7) / 8));
  if (a.sa_e8m0 && a.sb_e8m0)
    gemm_mid_kernel<C, true><<<grid, 64 * C::NW, 0, st>>>(a);
  else
    gemm_mid_kernel<C, false><<<grid, 64 * C::NW, 0, st>>>(a);
  return check_launch("gemm_mid");
}

}  // namespace

// The smallest tile, and so the most wavefronts per K block of it, that gives
// at most one workgroup per CU: a second round costs more than larger tiles
// (M = 1024, N = 4096 in two rounds of 64 x 128 tiles 52 us, 128 x 128 tiles 45).
int launch_dense_mid(GemmArgs& a, hipStream_t st) {
  const int64_t kb = a.K / 128, cus = device_cu_count();
  auto tiles = [&](int64_t bm, int64_t bn) { return ceil_div(a.M, bm) * ceil_div(a.N, bn); };
  if (kb <= 64 && tiles(32, 64) <= cus) return launch_mid<MidCfg<32, 64, 4, 3, 64>>(a, st);
  if (kb <= 64 && tiles(32, 128) <= cus) return launch_mid<MidCfg<32, 128, 2, 3, 64>>(a, st);
  // up to three tiles a CU where the 256 x 256 tiles that would take the
  // product (M > 2048) leave half the CUs or more without one: M = 4096, K =
  // 7168, those tiles / these, e8m0 and fp32 scales: N = 512 (one round) 84.1 /
  // 28.6 and 96.8 / 33.7 us, 1024 (two) 85.5 / 54.0 and 101 / 63.8, 1536 (three)
  // 89.9 / 81.0 and 106 / 92.8; K = 2048, N = 1536 35.0 / 30.7 and 38.6 / 34.7
  const bool few = a.M > 2048 && tiles(256, 256) <= cus / 2;
  if (kb <= 56 && tiles(64, 128) <= (few ? 3 * cus : cus)) return launch_mid<MidCfg<64, 128, 2, 3, 56>>(a, st);
  return kNoMid;
}

}  // namespace sgl
