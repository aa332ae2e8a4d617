// The routed + shared expert layer for the smallest batches (one to a few
// tokens): two launches after the activation quant instead of eight.
//
// At T = 1 a layer reads nine experts' weights once (132 MB with FP4 routed
// experts, 226 MB with FP8) and does almost nothing else, so what bounds it
// is how many CUs stream and how many launches stand between them.  The
// grouped GEMMs give a workgroup 256 columns of one expert (16 to 144
// workgroups a launch, each its 0.5-1 MB at one CU's rate) and need a
// permutation, a launch of its own for an FP4 layer's shared expert and a
// combine.  Here
//   gate/up  workgroup (16 gate + 16 up columns of one expert, FP8: 8 + 8):
//            finds its expert's rows by comparing the T k ids (no
//            permutation), sums its wavefronts' partials in LDS and stores
//            h = bf16(silu(gate) up w);
//   down     workgroup (16 output columns, every expert): quantizes the rows
//            of h into LDS, runs the picked experts and adds their bf16
//            outputs in ascending id, the shared one last, so y is written
//            by the workgroup that has every summand (no combine).
// Weights go to LDS by DMA in whole 128-byte lines (8 rows a 1 KB
// instruction), all of a wavefront's at once, and each wavefront computes the
// lines it fetched itself, so no barrier stands between a load and its MFMA.
// (Loaded straight into registers in the MFMA's lane order, half a line a
// row, the same split took 54 us for FP4 and 82 for FP8.)
// Numerics: the rounding points of the grouped path (bf16 gate and up, bf16
// h, 1x128 e4m3 h, bf16 expert outputs, fp32 sum in ascending expert id);
// each product's K is summed per line, then over lines in order.
//
// H = 4096, I = 2048, top-8 + shared, E = 256, one token, the layer with its
// activation quant, graph-replayed over cold weights: FP4 74.3 -> 41.3 us (gate/up
// 22.2, down 16.8 by the trace), FP8 65.5 -> 57.8 (32.1 and 22.4, where the two
// grouped launches took 33.0 and 20.3: only the permute and the combine are
// saved, so the rule small_moe_ok in sgl_rules.h ends early for FP8).
#include <algorithm>

#include "sgl_gemm.h"
#include "sgl_moe_small.h"
#include "sgl_numeric.h"

namespace sgl {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kMaxSlots = kSmallMoeSlots;

// One 128-deep K block of a row in MFMA lane order, lane group g: fp8 bytes
// [32 g, +32); the fp8 side of a product with fp4 bytes [16 g, +16) and
// [64 + 16 g, +16).
template <bool FP4>
__device__ __forceinline__ v8i load_a(const uint8_t* row, int g) {
  const uint4 lo = *reinterpret_cast<const uint4*>(row + (FP4 ? 16 : 32) * g);
  const uint4 hi = *reinterpret_cast<const uint4*>(row + (FP4 ? 16 * g + 64 : 32 * g + 16));
  return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

// A weight operand in LDS: 16 rows x one 128-byte line (fp8 a 128-deep K
// block, fp4 two), chunk c of row r at c ^ swz(r).
// Half q of it (rows 8 q ...) by one DMA: base + r * stride + line * 128.
__device__ __forceinline__ void dma_half(const uint8_t* base, int64_t stride, int line, int q, uint32_t lds,
                                         int lane) {
  const int rr = lane >> 3, pc = lane & 7;
  dma16v((uint64_t)(uintptr_t)base + (uint64_t)(rr * stride + line * 128) + (uint64_t)((pc ^ ((rr & 6) | q)) << 4),
         lds + (uint32_t)(q * 1024));
}
// K block sub of it as the MFMA's B operand (fp8: sub 0)
template <bool FP4>
__device__ __forceinline__ v8i read_w(const uint8_t* w, int sub, int g, int r) {
  const uint8_t* row = w + r * 128;
  if constexpr (FP4) {
    const uint4 v = *reinterpret_cast<const uint4*>(row + (((4 * sub + g) ^ swz(r)) << 4));
    return v8i{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
  } else {
    const uint4 lo = *reinterpret_cast<const uint4*>(row + (((2 * g) ^ swz(r)) << 4));
    const uint4 hi = *reinterpret_cast<const uint4*>(row + (((2 * g + 1) ^ swz(r)) << 4));
    return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  }
}

// acc += A . W^T of one K block, lane (g, r) holding rows 4 g + i, column r.
// sa: the scale of A row r (this lane's), the rows 4 g + i come from the
// lanes that hold them; sk: this column's fp8 block scale; sb: its four e8m0
// fp4 scales.
template <bool FP4>
__device__ __forceinline__ void mma(v4f& acc, const v8i& a, const v8i& b, float sa, float sk, uint32_t sb,
                                    bool pow2, int g) {
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (FP4) {
    const int s = (int)(sb >> (8 * g));
    if (pow2) {  // both scales as exponents inside the MFMA
      acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc, 0, 4, 0, (int)(f32_bits(sa) >> 23), 0, s);
      return;
    }
    const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, zero, 0, 4, 0, 127, 0, s);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(p[i], __shfl(sa, 4 * g + i, 64), acc[i]);
  } else {
    const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, zero, 0, 0, 0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(p[i], __shfl(sa, 4 * g + i, 64) * sk, acc[i]);
  }
}

// ---------------------------------------------------------------- gate / up
constexpr int kGuWaves = 8;
constexpr int kGuWaveLds = 8192;  // weight bytes of a wavefront at a time, then its partials

struct GuShared {
  alignas(16) uint8_t w[kGuWaves * kGuWaveLds];
  int slot[kMaxSlots];
};

// Columns [n0, n0 + NC) of gate and of up, NC = 16 (fp4: two operands) or 8
// (fp8: one operand, rows 0-7 gate and 8-15 up).
template <bool FP4>
__device__ __forceinline__ void gate_up_group(const SmallMoeArgs& a, GuShared& sm, const sgl_expert_ptrs* ex,
                                              int64_t n0, int nrows, bool shared) {
  constexpr int NC = FP4 ? 16 : 8;
  constexpr int NOP = FP4 ? 2 : 1;                      // operands per line
  constexpr int KPL = FP4 ? 2 : 1;                      // K blocks per line
  constexpr int NL = kGuWaveLds / (NOP * 2048);         // lines of a wavefront in LDS together
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, r16 = lane & 15;
  const int64_t H = a.H, I = a.I;
  const int KB = (int)(H / 128), lines = KB / KPL;
  const int64_t stride = FP4 ? H / 2 : H;
  const uint8_t* wg = (const uint8_t*)ex->w_gate + n0 * stride;
  const uint8_t* wu = (const uint8_t*)ex->w_up + n0 * stride;
  const uint8_t* sg = (const uint8_t*)ex->s_gate;
  const uint8_t* su = (const uint8_t*)ex->s_up;
  uint8_t* mine = sm.w + wave * kGuWaveLds;
  const uint32_t mine_lds = __builtin_amdgcn_readfirstlane(lds_u32(mine));
  for (int r0 = 0; r0 < nrows; r0 += 16) {
    if (r0 > 0) __syncthreads();  // the previous row tile's sums are read
    // this lane's A row; lanes past the last row hold zeros (their outputs are dropped)
    const bool row_ok = r0 + r16 < nrows;
    const int ri = row_ok ? r0 + r16 : r0;
    const int64_t t = shared ? ri : sm.slot[ri] / a.k;
    const uint8_t* arow = a.xq + t * H;
    const float* srow = a.xs + t * KB;
    v4f acc[NOP];
#pragma unroll
    for (int o = 0; o < NOP; ++o) acc[o] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (int l0 = wave; l0 < lines; l0 += kGuWaves * NL) {
      uint2 sw[NL][NOP];
      v8i af[NL][KPL];
      float sa[NL][KPL], sk[NL];
      if (l0 != wave) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last lines are read
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int line = l0 + kGuWaves * j;
        if (line < lines) {
          if constexpr (FP4) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              dma_half(wg + 8 * q * stride, stride, line, q, mine_lds + (2 * j) * 2048, lane);
              dma_half(wu + 8 * q * stride, stride, line, q, mine_lds + (2 * j + 1) * 2048, lane);
            }
          } else {
            dma_half(wg, stride, line, 0, mine_lds + j * 2048, lane);
            dma_half(wu, stride, line, 1, mine_lds + j * 2048, lane);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int line = l0 + kGuWaves * j;
        if (line < lines) {
          if constexpr (FP4) {
            sw[j][0] = *reinterpret_cast<const uint2*>(sg + (n0 + r16) * (H / 32) + line * 8);
            sw[j][NOP - 1] = *reinterpret_cast<const uint2*>(su + (n0 + r16) * (H / 32) + line * 8);
            sk[j] = 0.0f;
          } else {
            sk[j] = reinterpret_cast<const float*>(r16 < 8 ? sg : su)[(n0 / 128) * KB + line];
          }
#pragma unroll
          for (int sub = 0; sub < KPL; ++sub) {
            const int kb = line * KPL + sub;
            af[j][sub] = v8i{0, 0, 0, 0, 0, 0, 0, 0};
            sa[j][sub] = 0.0f;
            if (row_ok) {
              af[j][sub] = load_a<FP4>(arow + kb * 128, g4);
              sa[j][sub] = srow[kb];
            }
          }
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        if (l0 + kGuWaves * j < lines) {
#pragma unroll
          for (int sub = 0; sub < KPL; ++sub)
#pragma unroll
            for (int o = 0; o < NOP; ++o)
              mma<FP4>(acc[o], af[j][sub], read_w<FP4>(mine + (NOP * j + o) * 2048, sub, g4, r16), sa[j][sub], sk[j],
                       sub ? sw[j][o].y : sw[j][o].x, a.sa_pow2, g4);
        }
      }
    }
    // partials over this wavefront's weights: [row][operand][16 columns]
    float* red = reinterpret_cast<float*>(mine);
#pragma unroll
    for (int o = 0; o < NOP; ++o)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((4 * g4 + i) * NOP + o) * 16 + r16] = acc[o][i];
    __syncthreads();
    const int row = tid / NC, col = tid % NC;
    if (row < 16 && r0 + row < nrows) {
      float gs = 0.0f, us = 0.0f;
#pragma unroll
      for (int w = 0; w < kGuWaves; ++w) {
        const float* rw = reinterpret_cast<const float*>(sm.w + w * kGuWaveLds) + row * NOP * 16 + col;
        gs += rw[0];
        us += rw[FP4 ? 16 : 8];
      }
      float gt = bf16_round(gs), up = bf16_round(us);
      if (a.swiglu_limit > 0.0f) {
        up = clampf_(up, -a.swiglu_limit, a.swiglu_limit);
        gt = gt > a.swiglu_limit ? a.swiglu_limit : gt;
      }
      const float e = __builtin_amdgcn_exp2f(gt * -1.4426950408889634f);
      float h = gt * __builtin_amdgcn_rcpf(1.0f + e) * up;
      int64_t out = a.T * a.k + r0 + row;  // the shared rows follow the slots
      if (!shared) {
        out = sm.slot[r0 + row];
        h *= a.route_w[out];
      }
      a.h[out * I + n0 + col] = bf16_bits_exact(h);
    }
  }
}

// Workgroups: (slot, columns) of the routed experts, then the shared one's.
template <bool FP4>
__global__ __launch_bounds__(64 * kGuWaves) __attribute__((amdgpu_waves_per_eu(4, 4)))
void small_gate_up_kernel(const SmallMoeArgs a) {
  __shared__ GuShared sm;
  const int lane = threadIdx.x & 63;
  const int S = (int)(a.T * a.k);
  const int slabs = (int)(a.I / (FP4 ? 16 : 8));
  const int s = (int)blockIdx.x / slabs;
  if (s >= S) {  // the shared expert (always FP8), every token a row
    gate_up_group<false>(a, sm, a.experts + a.E, (int64_t)((int)blockIdx.x - S * slabs) * 8, (int)a.T, true);
    return;
  }
  const int e = a.ids[s];
  if (e < 0 || e >= a.E) return;
  const int id = lane < S ? a.ids[lane] : -1;
  const uint64_t m = __ballot(id == e);
  if (__builtin_ctzll(m) != s) return;  // the expert's first slot has its workgroups
  // every wavefront writes the whole list (the same values) and reads back its own writes
  if (id == e) sm.slot[__popcll(m & ((1ull << lane) - 1ull))] = lane;
  const int64_t n0 = (int64_t)((int)blockIdx.x - s * slabs) * (FP4 ? 16 : 8);
  gate_up_group<FP4>(a, sm, a.experts + e, n0, __popcll(m), false);
}

// --------------------------------------------------------------------- down
constexpr int kDnWaves = kSmallDownWaves;
constexpr int kDnLds = kSmallDownLds;  // (small_down_rows_bytes, then weights)

struct DnTables {
  int id[kMaxSlots];         // the slots' experts
  int slot[kMaxSlots];       // slots by (expert, slot)
  int tok[kMaxSlots];        // their tokens
  int start[kMaxSlots + 1];  // groups of equal expert in that order
  const uint8_t* w[kMaxSlots];  // the slots' w_down and s_down
  const uint8_t* s[kMaxSlots];
};

// The lines of K of `ng` groups' 16 weight rows, dealt to the wavefronts in
// turn; at most `slots` in a wavefront's LDS together.
template <bool FP4, bool SHARED>
__device__ __forceinline__ void down_groups(const SmallMoeArgs& a, const DnTables& tab, const uint8_t* hq,
                                            const float* hs, float* part, uint8_t* ring, int slots, int ng, int R,
                                            uint4 (&pre)[2]) {
  constexpr int KPL = FP4 ? 2 : 1;
  constexpr int NS = 5;  // slots at most
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g4 = lane >> 4, r16 = lane & 15;
  const int64_t I = a.I;
  const int KB = (int)(I / 128), lines = KB / KPL, tasks = ng * lines;
  const int64_t n0 = (int64_t)blockIdx.x * 16, stride = FP4 ? I / 2 : I;
  const int S = (int)(a.T * a.k);
  uint8_t* mine = ring + wave * slots * 2048;
  const uint32_t mine_lds = __builtin_amdgcn_readfirstlane(lds_u32(mine));
  const sgl_expert_ptrs* ex = a.experts + a.E;  // (read when there is a shared expert)
  const uint8_t* shared_w = a.has_shared ? (const uint8_t*)ex->w_down : nullptr;
  const uint8_t* shared_s = SHARED ? (const uint8_t*)ex->s_down : nullptr;
  uint2 sw[FP4 ? NS : 1];
  float sk[FP4 ? 1 : NS];
  auto fetch = [&](int t0) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last lines are read
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const int task = t0 + kDnWaves * j;
      if (j < slots && task < tasks) {
        const int g = task / lines, line = task - g * lines;
        const uint8_t* w = shared_w;
        const uint8_t* sc = shared_s;
        if constexpr (!SHARED) {
          const int s = tab.slot[tab.start[g]];
          w = tab.w[s];
          sc = tab.s[s];
        }
        w += n0 * stride;
        if (SHARED && task == wave) {  // fetched before the routed experts ran
          *reinterpret_cast<uint4*>(mine + j * 2048 + lane * 16) = pre[0];
          *reinterpret_cast<uint4*>(mine + j * 2048 + 1024 + lane * 16) = pre[1];
        } else {
#pragma unroll
          for (int q = 0; q < 2; ++q) dma_half(w + 8 * q * stride, stride, line, q, mine_lds + j * 2048, lane);
        }
        if constexpr (FP4)
          sw[j] = *reinterpret_cast<const uint2*>(sc + (n0 + r16) * (I / 32) + line * 8);
        else
          sk[j] = reinterpret_cast<const float*>(sc)[(n0 / 128) * KB + line];
      }
    }
  };
  fetch(wave);
  if constexpr (!SHARED) {
    if (a.has_shared && wave < KB) {  // line `wave` of the shared expert (FP8), in dma_half's order
      const int rr = lane >> 3, pc = lane & 7;
#pragma unroll
      for (int q = 0; q < 2; ++q)
        pre[q] = ld16_stream(shared_w + (n0 + 8 * q + rr) * I + wave * 128 + ((pc ^ ((rr & 6) | q)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // h is quantized (the loads stay in flight)
  }
  for (int t0 = wave; t0 < tasks; t0 += kDnWaves * slots) {
    if (t0 != wave) fetch(t0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const int task = t0 + kDnWaves * j;
      if (j < slots && task < tasks) {
        const int g = task / lines, line = task - g * lines;
        const int p0 = SHARED ? 0 : tab.start[g];
        const int nrows = SHARED ? (int)a.T : tab.start[g + 1] - p0;
        for (int r0 = 0; r0 < nrows; r0 += 16) {
          const int ri = min(r0 + r16, nrows - 1);
          const int row = SHARED ? S + ri : tab.slot[p0 + ri];
          v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int sub = 0; sub < KPL; ++sub) {
            const int kb = line * KPL + sub;
            mma<FP4>(acc, load_a<FP4>(hq + (int64_t)row * I + kb * 128, g4),
                     read_w<FP4>(mine + j * 2048, sub, g4, r16), hs[row * KB + kb], FP4 ? 0.0f : sk[FP4 ? 0 : j],
                     FP4 ? (sub ? sw[FP4 ? j : 0].y : sw[FP4 ? j : 0].x) : 0u, a.sa_pow2, g4);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int ro = r0 + 4 * g4 + i;
            if (ro < nrows) part[(line * R + (SHARED ? S + ro : tab.slot[p0 + ro])) * 16 + r16] = acc[i];
          }
        }
      }
    }
  }
}

template <bool FP4>
__global__ __launch_bounds__(64 * kDnWaves) void small_down_kernel(const SmallMoeArgs a, int slots) {
  __shared__ __align__(16) uint8_t buf[kDnLds];
  __shared__ DnTables tab;
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t I = a.I;
  const int KB = (int)(I / 128);
  const int T = (int)a.T, S = T * a.k, R = S + (a.has_shared ? T : 0);
  uint8_t* ring = buf;
  uint8_t* hq = buf + slots * kDnWaves * 2048;
  float* hs = reinterpret_cast<float*>(hq + (int64_t)R * I);
  float* part = hs + (int64_t)R * KB;

  // ---- the first rows of h on their way, 16 lanes a group of 128
  constexpr int NQ = 3;
  const int c = tid & 15;
  auto load_h = [&](int task) -> uint4 {
    const int row = task / KB, kb = task - row * KB;
    return *reinterpret_cast<const uint4*>(a.h + (int64_t)row * I + kb * 128 + 8 * c);
  };

  // ---- the slots by (expert, slot), those without a valid expert last; every
  // wavefront builds the same tables and reads back its own writes
  uint4 hv[NQ];
  int nvalid, ng;
  {
    const int v = lane < S ? a.ids[lane] : -1;
    const int id = v >= 0 && v < a.E ? v : 0x7FFFFFFF;
#pragma unroll
    for (int i = 0; i < NQ; ++i) hv[i] = load_h(min((tid >> 4) + 4 * kDnWaves * i, R * KB - 1));
    tab.id[lane] = id;
    nvalid = __popcll(__ballot(id != 0x7FFFFFFF));
    if (id != 0x7FFFFFFF) {
      tab.w[lane] = (const uint8_t*)a.experts[id].w_down;
      tab.s[lane] = (const uint8_t*)a.experts[id].s_down;
    }
    int rank = 0;
    for (int j0 = 0; j0 < S; j0 += 8) {  // (entries past S are no expert's)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int o = tab.id[j0 + j];
        rank += o < id || (o == id && j0 + j < lane);
      }
    }
    if (lane < S) {
      tab.slot[rank] = lane;
      tab.tok[rank] = lane / a.k;
    }
    const bool in = lane < nvalid;
    const int mine = in ? tab.id[tab.slot[lane]] : -1;
    const int before = __shfl_up(mine, 1, 64);  // (every lane takes part)
    const bool first = in && (lane == 0 || mine != before);
    const uint64_t m = __ballot(first);
    if (first) tab.start[__popcll(m & ((1ull << lane) - 1ull))] = lane;
    ng = __popcll(m);
    if (lane == 0) tab.start[ng] = nvalid;
  }

  // ---- h, bf16 -> e4m3 with 1x128 scales
  auto quant_h = [&](int task, const uint4& v) {
    const int row = task / KB, kb = task - row * KB;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    float f[8], amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = bits_f32(w[i] << 16);
      f[2 * i + 1] = bits_f32(w[i] & 0xFFFF0000u);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = __builtin_elementwise_maximum(amax, fabsf(f[i]));
    amax = lane_group_max<16>(amax);
    const float sf = group_scale(a.scale_mode, amax);
    *reinterpret_cast<uint2*>(hq + (int64_t)row * I + kb * 128 + 8 * c) = quant8_e4m3(a.scale_mode, f, sf);
    if (c == 0) hs[row * KB + kb] = sf;
  };
  for (int t0 = tid >> 4; t0 < R * KB; t0 += 4 * kDnWaves * NQ) {
    if (t0 != tid >> 4) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) hv[i] = load_h(min(t0 + 4 * kDnWaves * i, R * KB - 1));
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i)
      if (t0 + 4 * kDnWaves * i < R * KB) quant_h(t0 + 4 * kDnWaves * i, hv[i]);
  }

  // (the routed call holds the barrier behind h, after its first weights are on their way)
  uint4 pre[2] = {};
  down_groups<FP4, false>(a, tab, hq, hs, part, ring, slots, ng, R, pre);
  if (a.has_shared) down_groups<false, true>(a, tab, hq, hs, part, ring, slots, 1, R, pre);
  __syncthreads();
  // ---- a row's output: its lines' partials in order, rounded to bf16
  for (int i = tid; i < R * 16; i += 64 * kDnWaves) {
    const int lines = i < S * 16 && FP4 ? KB / 2 : KB;
    float v = 0.0f;
#pragma unroll 8
    for (int l = 0; l < lines; ++l) v += part[l * R * 16 + i];
    part[i] = bf16_round(v);
  }
  __syncthreads();
  // ---- a token's sum over its experts in ascending id, the shared one last
  for (int i = tid; i < T * 16; i += 64 * kDnWaves) {
    const int t = i >> 4, col = i & 15;
    float v = 0.0f;
#pragma unroll 8
    for (int p = 0; p < nvalid; ++p) {
      const float u = part[tab.slot[p] * 16 + col];
      if (tab.tok[p] == t) v += u;
    }
    if (a.has_shared) v += part[(S + t) * 16 + col];
    a.y[(int64_t)t * a.H + (int64_t)blockIdx.x * 16 + col] = bf16_bits_exact(v);
  }
}

}  // namespace

int launch_small_moe(const SmallMoeArgs& a, bool fp4, hipStream_t st) {
  const int64_t S = a.T * a.k, R = S + (a.has_shared ? a.T : 0);
  const unsigned gu = (unsigned)(S * (a.I / (fp4 ? 16 : 8)) + (a.has_shared ? a.I / 8 : 0));
  const unsigned dn = (unsigned)(a.H / 16);
  const int slots = std::min(5, small_down_slots(R, a.I));
  if (fp4) {
    small_gate_up_kernel<true><<<gu, 64 * kGuWaves, 0, st>>>(a);
    small_down_kernel<true><<<dn, 64 * kDnWaves, 0, st>>>(a, slots);
  } else {
    small_gate_up_kernel<false><<<gu, 64 * kGuWaves, 0, st>>>(a);
    small_down_kernel<false><<<dn, 64 * kDnWaves, 0, st>>>(a, slots);
  }
  return check_launch("moe_small");
}

}  // namespace sgl
