// Sparse multi-head attention over gathered KV rows: the MLA decode consumer
// of the packed FP8 KV cache.
//
// Semantics (deepseek_infer/kernel.py:276-368 sparse_attn_kernel): for every
// query token (b, m) and head h, over the rows kv[b, idx[b, m, j]] (j < K;
// idx = -1, or outside [0, n), is masked):
//     s_j = (q[h] . kv_j) * scale                       (bf16 x bf16, fp32 sum)
//     blocks of 64 rows, online:  m' = max(m, max_j s_j);  a = exp(m - m')
//         l = l a + sum_j exp(s_j - m');  o = o a + sum_j bf16(exp(s_j - m')) kv_j
//     o / (l + exp(sink[h] - m))  -> bf16
// The probabilities are cast to bf16 for the P.V product and summed in fp32
// for l, as the reference kernel does (the exponentials are taken base 2 on
// log2(e)-scaled scores, the same values up to fp32 rounding).  The KV rows
// are bf16, or the 584-byte layout A rows / footer pages of
// engine/dsv4_kv_pack.py dequantized on the way in (e4m3 * 2^(e8m0-127) is
// exact in bf16; v_cvt_scalef32_pk_bf16_fp8 rounds it exactly), so the packed
// cache feeds the attention with no bf16 copy of it in HBM.
//
// One workgroup per (query token, group of 64 heads, split of the indices); a
// small batch (decode) splits its indices over several workgroups, at most one
// a CU, and a second kernel merges the splits' partial maxima, sums and
// outputs (the rules, and the few heads and short chains that attn_few.hip
// takes: attn_plan in sgl_rules.h).  The split's valid indices are packed into
// a list in LDS first, so the masked entries of a call of one split (a
// prefill's early queries) cost only their index.  A split is a range of
// index positions: where they are all masked (the -1 pads at the end of a short
// context) its workgroup has no rows but still writes its partial.
// Eight wavefronts in two roles, one of each per SIMD, so one
// role's MFMAs fill the other's waits; the roles run blocks of 32 rows in
// phases with one barrier each, S^T of block j + 1 beside O^T of block j:
//   gather:  wavefronts 4-7, 8 rows each, into a ring of four 32 KB row-major
//            bf16 tiles: bf16 rows by LDS DMA two phases ahead; FP8 rows into
//            registers a phase ahead, then dequantized and stored;
//   S^T = KV . Q^T (v_mfma_f32_16x16x32_bf16), wavefronts 0-3: wavefront
//            (hh, th) 16 tokens x 32 heads over all 512 dims, its Q^T
//            fragments (128 registers) loaded once, so no partial sums meet;
//   P:       exp2 against the head's running reference, bf16, into one of two
//            4 KB LDS tiles.  The reference moves only when a score exceeds it
//            by more than 8 (log2 units), so as a rule no maxima are
//            exchanged: a wavefront that sees such a score raises a flag, and
//            only then the block's maxima meet in LDS and P and the
//            accumulators are brought to the new reference;
//   O^T += V^T . P^T (v_mfma_f32_32x32x16_bf16), wavefronts 4-7: wavefront w
//            128 dims of all 64 heads (128 registers), V^T fragments by
//            ds_read_b64_tr_b16 straight from the row-major tile, each of its
//            bytes read once.
// What bounds it: LDS traffic and MFMA issue, about evenly: per 32 rows the
// LDS takes 32 KB of tile writes, 64 KB of S^T reads, 32 KB (at half rate) of
// V^T reads and 16 KB of P reads; each SIMD 1024 cycles of MFMA (0.7 of the
// 1.1 us a block takes), and a workgroup fills a CU, so its first loads and
// its output rows (about 7 us a query) stand alone.  256 queries x 640 /
// 2048 rows of a bf16 cache 45.1 / 104 -> 34.0 / 73.6 us against the version
// before (one role, S^T over split dims with partial sums through LDS, 64-row
// blocks), packed pages 49.8 / 131 -> 37.7 / 92.2; a 2048-token prefill chunk
// (640 indices, -1 where a token has fewer rows) 321 -> 183 us.  The roles
// without the MFMAs between reads and gathers (each fragment read waited for
// by itself): 1.3 us a block.
#include "sgl_attn.h"
#include "sgl_numeric.h"

namespace sgl {
namespace {

// 16 bytes at an 8-byte aligned address (layout A rows)
typedef uint32_t V4a8 __attribute__((ext_vector_type(4), aligned(8)));

// A load from device memory at a 64-bit address: as a global load, since a flat
// one would count as LDS traffic too and be waited for at every barrier.
template <typename T>
__device__ __forceinline__ T ld_global(uint64_t addr) {
  typedef const T __attribute__((address_space(1))) gT;
  return *(gT*)(uintptr_t)addr;
}

// Barrier behind this wavefront's own LDS traffic and, with VM, its DMAs
// (which the compiler does not count).  The register loads the compiler
// counts stay in flight across the first form.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ void dma_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// dma16v when j < n: a branch inside the asm, so that the code around it
// stays one scheduling region.
__device__ __forceinline__ void dma16v_if(uint64_t addr, uint32_t lds, int j, int n) {
  asm volatile("s_cmp_ge_i32 %2, %3\n\ts_cbranch_scc1 .Lno_dma%=\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %0, off\n.Lno_dma%=:"
               :: "v"(addr), "s"(lds), "s"(j), "s"(n) : "memory", "scc");
}

constexpr int kRows = 32;            // rows of a block (one phase)
constexpr int kTile = kRows * 1024;  // bytes of a row-major bf16 tile
constexpr int kRing = 4;             // tiles
constexpr int kPTile = kHG * 64;     // bytes of P: [head][32 tokens] bf16

// Selected rows held in LDS at a time: their addresses and, FP8, the distance
// to their scale bytes.  A list that is not the last runs its whole blocks and
// leaves the rest to the next, so that the blocks (and with them the rounding)
// do not depend on its length.
template <int FMT>
constexpr int kList = FMT == SGL_ATTN_KV_BF16 ? 2752 : 1792;

template <int FMT>
struct Smem {
  alignas(16) uint8_t kv[kRing * kTile];  // row tiles (Q, then outputs, pass through them)
  alignas(16) uint8_t p[2 * kPTile];
  alignas(16) uint64_t row[kList<FMT> + kRows];
  uint32_t foot[FMT == SGL_ATTN_KV_BF16 ? 1 : kList<FMT> + kRows];
  float mx[2][kHG];                       // block maxima per token half and head (then the sums)
  float sink[kHG];                        // log2 units
  int flag[4];                            // block n's at n % 4: a score above its reference
  int64_t next;                           // index the next list starts at, -1: this is the last
};

__device__ const uint4 g_zero_row[64] = {};  // what a block's rows past the list read

// P [head h][32 tokens]: 16-byte chunk c (8 tokens) of row h.  The rotation
// spreads 16 heads' reads of one chunk over all 64 banks.
__device__ __forceinline__ uint32_t p_off(int h, int c) {
  return (uint32_t)(h * 64 + ((c ^ ((h >> 2) & 3)) << 4));
}

// One role of the workgroup: S (wavefronts 0-3: scores and probabilities) or
// not S (4-7: the outputs).  The two instantiations run the same sequence of
// barriers; keeping them apart keeps the 128 registers of Q^T and the 128 of
// O^T out of each other's wavefronts.
// HT: 32-head tiles of the group that exist (1: at most 32 heads in all).
template <int FMT, int HT, bool S>
__device__ __forceinline__ void attn_role(const AttnArgs& a, Smem<FMT>& sm) {
  constexpr bool kDma = FMT == SGL_ATTN_KV_BF16;
  uint8_t* const sKV = sm.kv;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hh = (wave >> 1) & 1, th = wave & 1;  // S: heads [32 hh, +32), tokens [16 th, +16)
  const int wo = wave & 3;                        // O: dims [128 wo, +128)
  const int l16 = lane & 15, g4 = lane >> 4;
  const int g2 = lane >> 5, c32 = lane & 31;
  const int64_t m = attn_query_in_seq(blockIdx.x, (uint32_t)a.M), b = blockIdx.y;
  const int split = (int)(blockIdx.z % a.nsplit);
  const int h0 = (int)(blockIdx.z / a.nsplit) * kHG;
  const int nh = min(a.Hh - h0, kHG);             // heads of this group
  const bool live = !S || 32 * hh < nh;           // S: this wavefront's heads exist
  const uint8_t* kvb = a.kv + b * a.kv_bstride;
  const int32_t* idxp = a.idx + (b * a.M + m) * a.K;
  const uint32_t kv_lds = __builtin_amdgcn_readfirstlane(lds_u32(sKV));

  // S^T operands: row l16 (a token, or a head), chunk 4 kk + g4; the swizzle
  // only touches the chunk's low four bits, so kk % 4 picks one of four bases
  // and the rest is an immediate offset
  uint32_t ka[4];
#pragma unroll
  for (int k4 = 0; k4 < 4; ++k4) ka[k4] = l16 * 1024 + (((4 * k4 + g4) ^ sw(l16)) << 4);
  // V^T operand by transpose read: in each 16-lane group G, source lane s
  // reads 4 dims of token 16 s4 + 8 (G >> 1) + 4 e + (s >> 2), and the read
  // hands each lane 4 consecutive tokens of one dim; e = 0, 1 give the lane's
  // 8 consecutive K elements.  Bases for each e; dim tile dt is chunk 4 dt of
  // the lane's low four chunk bits, which the swizzle only xors.
  uint32_t va[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int tok = 8 * (g4 >> 1) + 4 * e + (l16 >> 2);
    const int cl = 16 * wo + 2 * (g4 & 1) + ((l16 & 3) >> 1);
    va[e] = tok * 1024 + ((cl ^ sw(tok)) << 4) + 8 * (l16 & 1);
  }

  const float NEG_INF = -__builtin_huge_valf();
  const float c1 = a.scale * kLog2e;
  // reference points (log2 units): S: of heads 32 hh + 16 i + l16, with this
  // lane's share (its tokens) of their sums; O: of heads 32 i + c32
  float mref[2] = {NEG_INF, NEG_INF}, lsum[2] = {0.0f, 0.0f};
  // S: what the exponentials subtract (a fully masked prefix keeps o = 0) and
  // the raw score from which the reference has to move
  float nref[2] = {0.0f, 0.0f}, lim[2] = {NEG_INF, NEG_INF};
  v8bf qf[S ? 2 : 1][S ? 16 : 1];  // Q^T fragments: [head tile][32-dim step]
  v4f st[2];                       // S: scores of the last block
  v16f acc[S ? 1 : 4][S ? 1 : HT];  // O^T: [32-dim tile][32-head tile]
  if constexpr (!S) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int ht = 0; ht < HT; ++ht)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][ht][r] = 0.0f;
  }

  // the sinks, fetched long before they are used
  if (S && wave == 0 && lane < nh) sm.sink[lane] = a.sink[h0 + lane] * kLog2e;

  const int nblk_all = (int)((a.K + kBlk - 1) / kBlk);
  const int jb = split * a.bps;  // this split's first 64 indices
  const int64_t k_begin = (int64_t)jb * kBlk;
  const int64_t k_end = min((int64_t)min(jb + a.bps, nblk_all) * kBlk, a.K);

  int moves = 0;  // of the references
  bool first = true;
  for (int64_t kc = k_begin;;) {
    // ---- the valid rows from index kc on, packed in order, the last list
    // padded to a whole block.  Every wavefront writes the whole list (the same
    // values), so each reads back its own writes
    if (!first) __syncthreads();  // the previous list and tiles are consumed
    if (threadIdx.x < 4) sm.flag[threadIdx.x] = 0;
    int cnt = 0;
    auto put_row = [&](int at, int id) {
      if constexpr (kDma) {
        sm.row[at] = (uint64_t)(uintptr_t)kvb + (uint64_t)(uint32_t)id * ((uint64_t)a.ld * 2);
      } else if constexpr (FMT == SGL_ATTN_KV_A_PAGED) {
        const uint32_t pg = a.page_shift >= 0 ? (uint32_t)id >> a.page_shift : (uint32_t)id / (uint32_t)a.page;
        const uint32_t l = (uint32_t)id - pg * (uint32_t)a.page;
        sm.row[at] = (uint64_t)(uintptr_t)kvb + (uint64_t)pg * ((uint64_t)a.page * kARow) + l * (uint32_t)kAData;
        sm.foot[at] = (uint32_t)a.page * kAData - l * (uint32_t)(kAData - 8);
      } else {
        sm.row[at] = (uint64_t)(uintptr_t)kvb + (uint64_t)(uint32_t)id * kARow;
        sm.foot[at] = kAData;
      }
    };
    auto before = [](uint64_t mask) -> int {  // set bits below this lane
      return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
    };
    int64_t pe = kc;  // end of the indices taken
    int li = lane;  // made opaque, so that no address made from it is kept in registers across the phases
    asm volatile("" : "+v"(li));
    while (pe < k_end && cnt + 64 <= kList<FMT>) {
      int32_t id[4];
      const int64_t p0 = pe;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t p = p0 + u * 64 + li;
        id[u] = idxp[p < k_end ? p : k_end - 1];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (cnt + 64 > kList<FMT>) break;
        const bool ok = p0 + u * 64 + li < k_end && id[u] >= 0 && id[u] < a.n;
        const uint64_t mask = __ballot(ok);
        if (ok) put_row(cnt + before(mask), id[u]);
        cnt = __builtin_amdgcn_readfirstlane(cnt + __popcll(mask));
        pe = p0 + (u + 1) * 64;
      }
    }
    if (li < kRows) {  // (read only when cnt > 0: row 0 exists)
      if constexpr (kDma) sm.row[cnt + li] = (uint64_t)(uintptr_t)g_zero_row;
      else put_row(cnt + li, 0);
    }
    const bool last = pe >= k_end;
    const int nblk = (last ? cnt + kRows - 1 : cnt) / kRows;
    if (!last) {  // the next list starts at the first row left over
      int left = cnt - nblk * kRows;  // (a list that is not the last has more than a block)
      while (left > 0) {
        pe -= 64;
        const int32_t id = idxp[pe + li];
        const bool ok = id >= 0 && id < a.n;
        const uint64_t mask = __ballot(ok);
        const int here = __popcll(mask);
        if (here >= left) pe += __builtin_ctzll(__ballot(ok && before(mask) == here - left));
        left = here >= left ? 0 : left - here;
      }
    }
    sm.next = last ? -1 : pe;  // (kept here, not in the scalar registers, which the phases need)

    // ---- row gathers: rows 8 wo + rr of a block, by the O wavefronts (the
    // first time the S wavefronts take block 1).  bf16: one DMA per row, lane
    // i fetching the chunk that belongs at i.  FP8 (layout A): two rows a
    // load, 28 lanes each 16 e4m3 bytes (lanes 56-63 repeat lane 55) and
    // their scale byte, and one load for the 16-byte rope pieces of all eight
    // rows (lane: row lane / 8, piece lane % 8).  (One row a load, 56 lanes x
    // 8 bytes, with the scales passed between lanes, took three times the
    // instructions: 2048 rows x 256 queries 118 us against 105, both before
    // the loads were global ones)
    int ln = lane;  // made opaque where the gathers run, so that their per-row offsets are formed there
                    // and not kept in registers across the phases
    auto dma_row = [&](int j, int rr, uint64_t row) {  // (a block past the last: nothing)
      dma16v_if(row + (uint32_t)((ln ^ sw(8 * wo + rr)) << 4),
                kv_lds + (uint32_t)((j & (kRing - 1)) * kTile + wo * 8192 + rr * 1024), j, nblk);
    };
    struct Raw {  // FP8 rows on their way: two per pair
      V4a8 nope[kDma ? 1 : 4], rope;
      uint32_t sc[kDma ? 1 : 4];
    } raw;
    auto load_pair = [&](int at, int p, Raw& w) {
      const int lc = min(ln, 55), half = lc >= 28, piece = lc - 28 * half;
      const uint64_t row = sm.row[at + 2 * p + half];
      w.nope[p] = ld_global<V4a8>(row + 16 * piece);
      w.sc[p] = ld_global<uint8_t>(row + sm.foot[at + 2 * p + half] + (piece >> 2));
    };
    auto store_pair = [&](int j, int p, const Raw& w) {
      const int lc = min(ln, 55), half = lc >= 28, piece = lc - 28 * half;
      const uint32_t c = (uint32_t)(((2 * (p & 1)) << 2) | ((2 * wo + (p >> 1)) & 3));  // with half << 2: sw(row)
      const uint32_t off = (uint32_t)((j & (kRing - 1)) * kTile + wo * 8192 + p * 2048) +
                           ((uint32_t)(half * 1024 + ((2 * piece) ^ (half << 2)) * 16) ^ (c << 4));
      const float sc = bits_f32(w.sc[p] << 23);  // 2^(e8m0 - 127)
      const V4a8 x = w.nope[p];
      *reinterpret_cast<uint4*>(sKV + off) =
          make_uint4(cvt2_e4m3_bf16<false>(x.x, sc), cvt2_e4m3_bf16<true>(x.x, sc),
                     cvt2_e4m3_bf16<false>(x.y, sc), cvt2_e4m3_bf16<true>(x.y, sc));
      *reinterpret_cast<uint4*>(sKV + (off ^ 16)) =
          make_uint4(cvt2_e4m3_bf16<false>(x.z, sc), cvt2_e4m3_bf16<true>(x.z, sc),
                     cvt2_e4m3_bf16<false>(x.w, sc), cvt2_e4m3_bf16<true>(x.w, sc));
    };
    auto load_rope = [&](int at) -> V4a8 { return ld_global<V4a8>(sm.row[at + (ln >> 3)] + kANope + 16 * (ln & 7)); };
    auto store_rope = [&](int j, const V4a8& x) {  // then zeros for the rows past the list
      const int t = 8 * wo + (ln >> 3);
      uint8_t* tile = sKV + (j & (kRing - 1)) * kTile;
      *reinterpret_cast<uint4*>(tile + t * 1024 + (((56 + (ln & 7)) ^ sw(t)) << 4)) = make_uint4(x.x, x.y, x.z, x.w);
      const int left = cnt - j * kRows - 8 * wo;
      if (left < 8)
        for (int rr = max(left, 0); rr < 8; ++rr)
          *reinterpret_cast<uint4*>(tile + (8 * wo + rr) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
    };
    asm volatile("" : "+v"(ln));
    {
      const int j = S ? 1 : 0, at = j * kRows + 8 * wo;
      if (j < nblk) {
        if constexpr (kDma) {
#pragma unroll
          for (int rr = 0; rr < 8; ++rr) dma_row(j, rr, sm.row[at + rr]);
        } else {
#pragma unroll
          for (int p = 0; p < 4; ++p) load_pair(at, p, raw);
          raw.rope = load_rope(at);
        }
      }
      if (first) {
        // Q rows through the last two tiles: one DMA per head row
#pragma unroll
        for (int rr = 0; rr < 8; ++rr) {
          const int h = 8 * wave + rr;
          const uint8_t* row = reinterpret_cast<const uint8_t*>(
              a.q + ((b * a.M + m) * a.Hh + h0 + min(h, nh - 1)) * (int64_t)kD);
          dma16(row, (uint32_t)((lane ^ sw(h)) << 4), kv_lds + (uint32_t)(2 * kTile + h * 1024));
        }
      }
      if constexpr (!kDma) {
        if (j < nblk) {
#pragma unroll
          for (int p = 0; p < 4; ++p) store_pair(j, p, raw);
          store_rope(j, raw.rope);
        }
      }
    }
    dma_barrier();  // tiles 0 and 1, and Q, are whole
    if (first) {
      if constexpr (S) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int kk = 0; kk < 16; ++kk)
            qf[i][kk] = *reinterpret_cast<const v8bf*>(sKV + 2 * kTile + (32 * hh + 16 * i) * 1024 +
                                                       ka[kk & 3] + 256 * (kk >> 2));
      }
      lds_barrier();  // Q is out of the tiles
      first = false;
    }

    // S: P of this lane's tokens of block n against the current references
    float ls[2] = {0.0f, 0.0f};
    auto put_p = [&](int n) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[i][r], c1, nref[i]));
        ls[i] = (p[0] + p[1]) + (p[2] + p[3]);
        *reinterpret_cast<uint2*>(sm.p + (n & 1) * kPTile + p_off(32 * hh + 16 * i + l16, 2 * th + (g4 >> 1)) +
                                  8 * (g4 & 1)) = make_uint2(pk2_bf16(p[0], p[1]), pk2_bf16(p[2], p[3]));
      }
    };
    // Block n has a score above its head's reference: the reference of a head
    // moves to its block maximum where that exceeds it by more than 8 (log2
    // units; the second time by anything, since the largest probability, 1,
    // is exact in bf16 and the first 32 rows hold it less often): the
    // probabilities stay <= 256 (exact range in bf16, same relative rounding).
    // Any reference gives the same softmax.  Both roles come here, the S
    // wavefronts with block n's scores in st.
    auto put_max = [&]() {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float mx = __builtin_fmaxf(__builtin_fmaxf(st[i][0], st[i][1]), __builtin_fmaxf(st[i][2], st[i][3]));
        mx = __builtin_fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = __builtin_fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (g4 == 0) sm.mx[th][32 * hh + 16 * i + l16] = mx;
      }
    };
    auto move_refs = [&](int n) {
      if (moves > 0) {  // (the first block leaves its maxima, and no P)
        if constexpr (S) {
          if (live) put_max();
        }
        lds_barrier();  // maxima exchanged
      }
      const float slack = moves < 2 ? 0.0f : 8.0f;
      ++moves;
      float f[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int h = S ? 32 * hh + 16 * i + l16 : 32 * i + c32;
        const float mx = __builtin_fmaxf(sm.mx[0][h], sm.mx[1][h]) * c1;  // (scale > 0)
        const float mn = !(mx <= mref[i] + slack) ? __builtin_fmaxf(mref[i], mx) : mref[i];
        f[i] = mn == mref[i] ? 1.0f : __builtin_amdgcn_exp2f(mref[i] - (mn == NEG_INF ? 0.0f : mn));
        mref[i] = mn;
      }
      if constexpr (S) {
        if (live) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            lsum[i] *= f[i];
            nref[i] = mref[i] == NEG_INF ? 0.0f : -mref[i];
            lim[i] = (mref[i] + (moves < 2 ? 0.0f : 8.0f)) / c1;
          }
          put_p(n);
        }
      } else {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int ht = 0; ht < HT; ++ht)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[dt][ht][r] *= f[ht];
      }
      lds_barrier();  // P rewritten
    };

    // ---- phases: in phase j S^T and P of block j + 1 beside O^T of block j,
    // one barrier after each.  A phase's first reads go out before the flag of
    // block j is looked at
    if constexpr (S) {
      for (int j = -1; j < nblk; ++j) {
        const int n = j + 1;
        const uint8_t* tile = sKV + (n & (kRing - 1)) * kTile + 16 * th * 1024;
        // four groups of four 32-dim steps, each group's fragments read while
        // the one before is multiplied (left to itself the compiler reads one
        // fragment, waits for it and multiplies)
        v8bf kvf[2][4];
        auto read4 = [&](int g) {
#pragma unroll
          for (int k4 = 0; k4 < 4; ++k4)
            kvf[g & 1][k4] = *reinterpret_cast<const v8bf*>(tile + ka[k4] + 256 * g);
        };
        const int flag = sm.flag[j & 3];
        read4(0);
        __builtin_amdgcn_sched_barrier(0);
        if (j >= 0) {
          if (__builtin_amdgcn_readfirstlane(flag)) move_refs(j);
          lsum[0] += ls[0];
          lsum[1] += ls[1];
        }
        if (threadIdx.x == 0) sm.flag[(j + 2) & 3] = 0;
        if (n < nblk && live) {
          // lane (head l16, g4) gets tokens 16 th + 4 g4 + r
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) st[i][r] = 0.0f;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            if (g < 3) read4(g + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
              for (int i = 0; i < 2; ++i)
                st[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kvf[g & 1][k4], qf[i][4 * g + k4], st[i], 0, 0, 0);
          }
          if (cnt - n * kRows < kRows) {
            const int left = cnt - n * kRows - 16 * th - 4 * g4;  // this lane's tokens past it are masked
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (r >= left) st[0][r] = st[1][r] = NEG_INF;
          }
          bool over = moves == 0;
#pragma unroll
          for (int i = 0; i < 2; ++i)
            over |= !(__builtin_fmaxf(__builtin_fmaxf(st[i][0], st[i][1]),
                                      __builtin_fmaxf(st[i][2], st[i][3])) <= lim[i]);
          if (__ballot(over) && lane == 0) sm.flag[n & 3] = 1;
          if (moves == 0) put_max();
          else put_p(n);
        }
        lds_barrier();
      }
    } else {
      // the rows of block 2
      uint64_t row_next[kDma ? 8 : 1];  // bf16: the addresses of the next eight rows
      auto list_at = [&](int j) -> int { return min(j, nblk - 1) * kRows + 8 * wo; };
      auto read_rows = [&](int j) {
        if constexpr (kDma) {
#pragma unroll
          for (int rr = 0; rr < 8; rr += 2) {
            const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(&sm.row[list_at(j) + rr]);
            row_next[rr] = v.x;
            row_next[rr + 1] = v.y;
          }
        }
      };
      if (nblk > 0) {
        read_rows(2);
        if constexpr (kDma) {
#pragma unroll
          for (int rr = 0; rr < 8; ++rr) dma_row(2, rr, row_next[rr]);
        } else {
#pragma unroll
          for (int p = 0; p < 4; ++p) load_pair(list_at(2), p, raw);
          raw.rope = load_rope(list_at(2));
        }
      }
      lds_barrier();  // (block 1's tile, the first time whole, is S's next)
      for (int j = 0; j < nblk; ++j) {
        const uint8_t* tile = sKV + (j & (kRing - 1)) * kTile;
        v8bf pf[2][HT], vf[2][4];
        auto read_p = [&](int s4) {
#pragma unroll
          for (int ht = 0; ht < HT; ++ht)
            pf[s4][ht] = *reinterpret_cast<const v8bf*>(sm.p + (j & 1) * kPTile + p_off(32 * ht + c32, 2 * s4 + g2));
        };
        auto read_v = [&](int s4) {
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            const v4s lo = lds_tr16(tile, (va[0] ^ (dt << 6)) + 16384 * s4);
            const v4s hi = lds_tr16(tile, (va[1] ^ (dt << 6)) + 16384 * s4);
            vf[s4][dt] = __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          }
        };
        const int flag = sm.flag[j & 3];
        if constexpr (!kDma) asm volatile("" : "+v"(va[0]), "+v"(va[1]));  // (the eight addresses: not kept)
        read_p(0);
        read_v(0);
        read_rows(j + 3);
        __builtin_amdgcn_sched_barrier(0);
        if (__builtin_amdgcn_readfirstlane(flag)) {
          move_refs(j);
          read_p(0);
        }
        if constexpr (kDma) {  // (FP8: below, for want of registers)
          read_p(1);
          read_v(1);
        }
        asm volatile("" : "+v"(ln));
        __builtin_amdgcn_sched_barrier(0);
        // the MFMAs, and between them the gathers: bf16: block j + 3's DMAs,
        // into the tile that held block j - 1; FP8: block j + 2's rows, loaded
        // during the last phase, dequantized into their tile (past the last
        // block, into a tile nobody reads), then block j + 3's loads
#pragma unroll
        for (int rr = 0; rr < 8; ++rr) {
          const int s4 = rr >> 2, dt = rr & 3;
          if constexpr (kDma) {
            dma_row(j + 3, rr, row_next[rr]);
          } else {
            if (rr == 2) {
              read_p(1);
              read_v(1);
            }
            if (rr & 1)
              load_pair(list_at(j + 3), rr >> 1, raw);
            else
              store_pair(j + 2, rr >> 1, raw);
          }
#pragma unroll
          for (int ht = 0; ht < HT; ++ht)
            acc[dt][ht] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[s4][dt], pf[s4][ht], acc[dt][ht], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!kDma) {
          store_rope(j + 2, raw.rope);
          raw.rope = load_rope(list_at(j + 3));
        }
        // block j + 2's tile whole (block j + 3's eight DMAs may be in flight)
        if constexpr (kDma) {
          if (j + 3 < nblk)
            asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
          else
            dma_barrier();
        } else {
          lds_barrier();
        }
      }
    }
    const int2 next = *reinterpret_cast<const int2*>(&sm.next);
    const int next_hi = __builtin_amdgcn_readfirstlane(next.y);
    if (next_hi < 0) break;
    kc = (int64_t)next_hi << 32 | (uint32_t)__builtin_amdgcn_readfirstlane(next.x);
  }

  // ---- the heads' sums meet in LDS; the outputs pass through the tiles so
  // that they leave as whole rows
  __syncthreads();
  if constexpr (S) {
    if (live) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float l = lsum[i];
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        if (g4 == 0) sm.mx[th][32 * hh + 16 * i + l16] = l;
      }
    }
  }
  __syncthreads();
  const int64_t qm = b * a.M + m;
  if constexpr (!S) {
    // lane (head 32 ht + c32, g2) holds dims 128 wo + 32 dt + 8 q4 + 4 g2 + 0..3
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      const int h = 32 * ht + c32;
      if (h < nh) {
        const float l = sm.mx[0][h] + sm.mx[1][h];
        if (a.nsplit > 1) {
          if (wo == 0 && g2 == 0) {
            float* ml = a.ws_ml + ((qm * a.nsplit + split) * a.Hh + h0 + h) * 2;
            ml[0] = mref[ht];
            ml[1] = l;
          }
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
              const int c = 32 * wo + 8 * dt + 2 * q4 + g2;
              *reinterpret_cast<float4*>(sKV + h * 2048 + ((c ^ sw(h)) << 4)) =
                  make_float4(acc[dt][ht][4 * q4], acc[dt][ht][4 * q4 + 1], acc[dt][ht][4 * q4 + 2],
                              acc[dt][ht][4 * q4 + 3]);
            }
        } else {
          // o = acc / (l + exp(sink - m))
          const float ref = mref[ht] == NEG_INF ? 0.0f : mref[ht];
          const float inv = 1.0f / (l + __builtin_amdgcn_exp2f(sm.sink[h] - ref));
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
              const int c = 16 * wo + 4 * dt + q4;
              *reinterpret_cast<uint2*>(sKV + h * 1024 + ((c ^ sw(h)) << 4) + 8 * g2) =
                  make_uint2(pk2_bf16(acc[dt][ht][4 * q4] * inv, acc[dt][ht][4 * q4 + 1] * inv),
                             pk2_bf16(acc[dt][ht][4 * q4 + 2] * inv, acc[dt][ht][4 * q4 + 3] * inv));
            }
        }
      }
    }
  }
  __syncthreads();
  for (int h = wave; h < nh; h += 8) {
    if (a.nsplit > 1) {
      float* row = a.ws_acc + ((qm * a.nsplit + split) * a.Hh + h0 + h) * (int64_t)kD;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int c = 64 * u + lane;
        *reinterpret_cast<float4*>(row + 4 * c) =
            *reinterpret_cast<const float4*>(sKV + h * 2048 + ((c ^ sw(h)) << 4));
      }
    } else {
      uint16_t* row = a.o + (qm * a.Hh + h0 + h) * (int64_t)kD;
      *reinterpret_cast<uint4*>(row + 8 * lane) =
          *reinterpret_cast<const uint4*>(sKV + h * 1024 + ((lane ^ sw(h)) << 4));
    }
  }
}

template <int FMT, int HT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void sparse_attn_kernel(const AttnArgs a) {
  __shared__ Smem<FMT> sm;
  static_assert(sizeof(sm) <= 160 * 1024, "the LDS of a CU");
  if (threadIdx.x < 256)
    attn_role<FMT, HT, true>(a, sm);
  else
    attn_role<FMT, HT, false>(a, sm);
}

// Merge of the per-split partials, one wavefront per (query, head), maxima in
// log2 units:
//   M = max_s m_s;  o = sum_s acc_s 2^(m_s - M) / (sum_s l_s 2^(m_s - M) + e^(sink) 2^(-M))
// (splits whose rows were all masked carry m = -inf and add nothing).
__global__ __launch_bounds__(256) void sparse_attn_combine_kernel(const AttnArgs a, uint32_t queries) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const AttnMerge at = attn_merge_at(blockIdx.x, wave, queries, (uint32_t)a.M, (uint32_t)a.Hh);
  if (at.query >= queries || at.head >= (uint32_t)a.Hh) return;
  const int64_t q = at.query;  // b * M + m
  const int h = (int)at.head;
  const int64_t w = q * a.Hh + h;
  const float NEG_INF = -__builtin_huge_valf();
  // every split's loads are issued before the first is used (at most
  // kAttnMaxSplits splits), so their latencies overlap instead of adding up;
  // the maximum and the sums then run in split order as before
  float msp[kAttnMaxSplits], lsp[kAttnMaxSplits];
  float4 usp[kAttnMaxSplits], vsp[kAttnMaxSplits];
#pragma unroll
  for (int sp = 0; sp < kAttnMaxSplits; ++sp) {
    if (sp < a.nsplit) {
      const int64_t r = (q * a.nsplit + sp) * a.Hh + h;
      msp[sp] = a.ws_ml[r * 2];
      lsp[sp] = a.ws_ml[r * 2 + 1];
      const float4* src = reinterpret_cast<const float4*>(a.ws_acc + r * kD + lane * 8);
      usp[sp] = src[0];
      vsp[sp] = src[1];
    }
  }
  float mx = NEG_INF;
#pragma unroll
  for (int sp = 0; sp < kAttnMaxSplits; ++sp)
    if (sp < a.nsplit) mx = fmaxf_(mx, msp[sp]);
  const float ref = mx == NEG_INF ? 0.0f : mx;
  float o[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  float l = 0.0f;
#pragma unroll
  for (int sp = 0; sp < kAttnMaxSplits; ++sp) {
    if (sp < a.nsplit) {
      const float f = __builtin_amdgcn_exp2f(msp[sp] - ref);  // 0 for an all-masked split
      l += lsp[sp] * f;
      const float4 u = usp[sp], v = vsp[sp];
      o[0] += u.x * f; o[1] += u.y * f; o[2] += u.z * f; o[3] += u.w * f;
      o[4] += v.x * f; o[5] += v.y * f; o[6] += v.z * f; o[7] += v.w * f;
    }
  }
  const float den = l + __builtin_amdgcn_exp2f(a.sink[h] * kLog2e - ref);
  uint32_t wv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wv[i] = pk2_bf16_exact(o[2 * i] / den, o[2 * i + 1] / den);
  *reinterpret_cast<uint4*>(a.o + w * (int64_t)kD + lane * 8) = make_uint4(wv[0], wv[1], wv[2], wv[3]);
}

}  // namespace
}  // namespace sgl

extern "C" size_t sgl_sparse_attn_workspace_size(int64_t B, int64_t M, int Hh, int64_t K) {
  if (B <= 0 || M <= 0 || Hh <= 0 || K <= 0) return 0;
  const int ns = sgl::attn_plan(B * M, Hh, K, sgl::device_cu_count()).nsplit;
  if (ns == 1) return 0;
  return (size_t)(B * M * ns * Hh) * (sgl::kD + 2) * 4;
}

extern "C" int sgl_sparse_attn(const void* q, int64_t B, int64_t M, int Hh, const void* kv,
                               int kv_format, int page_size, int64_t n, int64_t kv_batch_stride,
                               int64_t ld, const float* attn_sink, const int32_t* topk_idxs,
                               int64_t K, float softmax_scale, void* o, void* workspace,
                               size_t workspace_bytes, sgl_stream_t stream) {
  SGL_REQUIRE(B >= 0 && M >= 0 && K >= 0 && n >= 0 && Hh >= 1, "sparse_attn: bad sizes");
  SGL_REQUIRE(softmax_scale > 0.0f, "sparse_attn: softmax_scale must be positive");
  SGL_REQUIRE(kv_format == SGL_ATTN_KV_BF16 || kv_format == SGL_ATTN_KV_A ||
                  kv_format == SGL_ATTN_KV_A_PAGED,
              "sparse_attn: bad kv_format %d", kv_format);
  SGL_REQUIRE(kv_format != SGL_ATTN_KV_A_PAGED || page_size > 0, "sparse_attn: page_size must be positive");
  SGL_REQUIRE(kv_format != SGL_ATTN_KV_BF16 || ld >= 512, "sparse_attn: bf16 kv row stride %lld < 512",
              (long long)ld);
  if (B == 0 || M == 0) return SGL_OK;
  SGL_REQUIRE(q && kv && attn_sink && o && (K == 0 || topk_idxs), "sparse_attn: null pointer");
  SGL_REQUIRE(sgl::aligned(q, 16) && sgl::aligned(o, 16) &&
                  sgl::aligned(kv, kv_format == SGL_ATTN_KV_BF16 ? 16 : 8) &&
                  (kv_format != SGL_ATTN_KV_BF16 || (ld % 8 == 0 && kv_batch_stride % 16 == 0)) &&
                  kv_batch_stride % 8 == 0,
              "sparse_attn: misaligned q / kv");
  SGL_REQUIRE(M <= 0x7FFFFFFF && B <= 65535, "sparse_attn: grid too large");
  sgl::AttnArgs a;
  a.q = (const uint16_t*)q;
  a.kv = (const uint8_t*)kv;
  a.n = n;
  a.kv_bstride = kv_batch_stride;
  a.ld = ld;
  a.page = page_size;
  a.page_shift = (page_size > 0 && (page_size & (page_size - 1)) == 0) ? __builtin_ctz((unsigned)page_size) : -1;
  a.sink = attn_sink;
  a.idx = topk_idxs;
  a.M = M;
  a.K = K;
  a.Hh = Hh;
  a.scale = softmax_scale;
  a.o = (uint16_t*)o;
  const sgl::AttnPlan plan = sgl::attn_plan(B * M, Hh, K, sgl::device_cu_count());
  a.nsplit = plan.nsplit;
  const int64_t nblk = (K + sgl::kBlk - 1) / sgl::kBlk;
  a.bps = (int)((nblk + a.nsplit - 1) / a.nsplit);
  a.ws_acc = nullptr;
  a.ws_ml = nullptr;
  if (a.nsplit > 1) {
    const size_t need = sgl_sparse_attn_workspace_size(B, M, Hh, K);
    if (workspace_bytes < need || !workspace) {
      sgl::set_error("sparse_attn: workspace %zu bytes < %zu needed", workspace_bytes, need);
      return SGL_ERR_WORKSPACE;
    }
    SGL_REQUIRE(sgl::aligned(workspace, 16), "sparse_attn: workspace must be 16-byte aligned");
    a.ws_acc = (float*)workspace;
    a.ws_ml = a.ws_acc + B * M * a.nsplit * (int64_t)Hh * sgl::kD;
  }
  dim3 grid((unsigned)M, (unsigned)B, (unsigned)(((Hh + sgl::kHG - 1) / sgl::kHG) * a.nsplit));
  hipStream_t st = (hipStream_t)stream;
  const bool one = Hh <= 32;  // (a last group of at most 32 heads beside full ones computes both tiles)
#define SGL_ATTN(FMT)                                                   \
  do {                                                                  \
    if (one)                                                            \
      sgl::sparse_attn_kernel<FMT, 1><<<grid, 512, 0, st>>>(a);         \
    else                                                                \
      sgl::sparse_attn_kernel<FMT, 2><<<grid, 512, 0, st>>>(a);         \
  } while (0)
  if (plan.few)
    sgl::launch_sparse_attn_few(a, kv_format, grid, st);
  else if (kv_format == SGL_ATTN_KV_BF16)
    SGL_ATTN(SGL_ATTN_KV_BF16);
  else if (kv_format == SGL_ATTN_KV_A)
    SGL_ATTN(SGL_ATTN_KV_A);
  else
    SGL_ATTN(SGL_ATTN_KV_A_PAGED);
#undef SGL_ATTN
  if (a.nsplit > 1) {
    // (more than one split: fewer queries x head groups than CUs)
    const uint32_t Q = (uint32_t)(B * M);
    sgl::sparse_attn_combine_kernel<<<sgl::attn_merge_groups(Q, (uint32_t)Hh), 256, 0, st>>>(a, Q);
  }
  return sgl::check_launch("sparse_attn");
}
