// Size rules of the dispatches: which query, kernel, tile or split a launch
// takes, as functions of its sizes (and of the device's CU count) alone.
// Plain C++ without HIP, so that a host test can walk over them.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define SGL_RULE __host__ __device__ inline
#else
#define SGL_RULE inline
#endif

namespace sgl {

// ---- sparse attention: the order of the queries.  The grid's launch index is
// i = blockIdx.x + M blockIdx.y; the later queries of a sequence, which select
// more rows in a prefill, start first.
SGL_RULE uint32_t attn_query_in_seq(uint32_t x, uint32_t M) { return M - 1 - x; }
SGL_RULE uint32_t attn_query_at(uint32_t i, uint32_t M) {
  const uint32_t b = i / M;
  return b * M + attn_query_in_seq(i - b * M, M);
}

// The merge of a query's splits, one wavefront per (query, head), four a
// workgroup.  Workgroups go round the eight XCDs in order, so with a multiple
// of eight queries every split of the query at launch index i ran on XCD i % 8,
// and the merge's workgroup goes there too and finds the partials in that L2
// (32 sequences x 640 rows: the attention kernel 21.9 -> 19.2 us, as its
// partial lines stay with one L2, the merge 5.4 -> 4.3; 4 sequences of 8
// queries, merged on another XCD 30.4 us a call, so 22.8).  With any other
// count the splits of a query are spread over XCDs, and the order is plain.
struct AttnMerge {
  uint32_t query, head;  // past the last: no work
};
SGL_RULE uint32_t attn_merge_groups(uint32_t queries, uint32_t heads) {
  return queries % 8 == 0 ? queries * ((heads + 3) / 4) : (queries * heads + 3) / 4;
}
SGL_RULE AttnMerge attn_merge_at(uint32_t wg, uint32_t wave, uint32_t queries, uint32_t M, uint32_t heads) {
  if (queries % 8 == 0) {
    const uint32_t per = (heads + 3) / 4, i = wg >> 3;
    const uint32_t at = 8 * (i / per) + (wg & 7);
    return {at < queries ? attn_query_at(at, M) : queries, 4 * (i % per) + wave};
  }
  const uint32_t w = 4 * wg + wave;
  return {w / heads, w % heads};
}

// ---- sparse attention: the kernel, and the workgroups (splits) that share a
// query's K indices, cut in 64s: at most one a CU, at most kAttnMaxSplits.  A
// function of the shape alone and not of the cache's format, so that the packed
// cache gives bit for bit what its dequantized rows give.
//
// A split shortens the serial chain of blocks but writes fp32 partials (128 KB
// per 64 heads) that a merge reads back; attn_few.hip (at most 64 heads) starts
// sooner than attn.hip but is slower a block.  The cheapest by these costs, in
// 1/100 us, fitted to 1 ... 256 queries x 64 ... 2048 indices x 1 ... 128 heads,
// all valid, bf16 rows and packed pages, both kernels, every number of splits
// (the choice is within 0.4 % of the best for each shape and format on average;
// one choice for both formats costs bf16 rows up to about 13 %):
//   a block of 64 indices: 250 (attn.hip, whose own blocks are 32 rows: at most
//     32 indices 125);
//   attn_few.hip against attn.hip: 75 a block more, and to start 288 - 4 heads
//     less (at most 32 heads) or 185 - 4.7 (heads - 32) less;
//   a merge: 250 and 31 a split, up to 74 more with the heads, and for each
//     partial of 64 heads 4.5 where the merge follows its splits (a multiple of
//     eight queries), else 8, at most 900.
// (Packed pages, us.  64 heads: 32 / 33 queries x 128 indices, one split / two
// 15.2 / 17.4 and 15.1 / 20.7; 32 x 384, one / three 25.3 / 20.8; 32 x 640, one
// / five 35.6 / 23.5; 33 x 2048, seven 36.7, eight, which are 264 workgroups,
// 52.6.  256 queries, few / attn.hip: 8 heads x 64 indices 9.3 / 12.2, x 192
// 16.1 / 17.0, x 640 38.7 / 36.9; 32 heads 12.3 / 14.1, 19.1 / 18.9, 41.3 /
// 38.6; one query x 8 heads x 256, four splits 10.8 / 13.5, x 32 heads x 1 index
// 9.2 / 8.5.)
constexpr int kAttnMaxSplits = 8;
struct AttnPlan {
  bool few;  // attn_few.hip
  int nsplit;
};
SGL_RULE AttnPlan attn_plan(int64_t queries, int heads, int64_t K, int cus) {
  const int64_t blocks = (K + 63) / 64, wgs = queries * ((heads + 63) / 64);
  const int64_t h64 = heads < 64 ? heads : 64;
  AttnPlan best = {false, 1};
  int64_t best_cost = K <= 32 ? 125 : blocks * 250;
  for (int kernel = 0; kernel < (heads <= 64 ? 2 : 1); ++kernel) {
    const bool few = kernel == 1;
    const int64_t start = !few ? 0 : heads <= 32 ? 288 - 4 * heads : 185 - 47 * (heads - 32) / 10;
    for (int64_t want = 1; want <= kAttnMaxSplits && (want == 1 || (want <= blocks && want * wgs <= cus)); ++want) {
      const int64_t bps = (blocks + want - 1) / want;
      const int64_t ns = bps > 0 ? (blocks + bps - 1) / bps : 1;  // no empty split
      int64_t cost = (!few && K <= 32 ? 125 : bps * (few ? 325 : 250)) - start;
      if (ns > 1) {
        int64_t parts = queries * ns * heads * (queries % 8 == 0 ? 45 : 80) / 640;
        if (queries % 8 != 0 && parts > 900) parts = 900;
        cost += 250 + 31 * ns + 74 * h64 / 64 + parts;
      }
      if (cost < best_cost) {
        best_cost = cost;
        best = {few, (int)ns};
      }
    }
  }
  return best;
}

// ---- dense FP8 GEMM, 16 < M <= 64: the tiles that split K inside a workgroup
// (dense_mid.hip) against the split over workgroups (`splits`: the shape has
// one) or else the skinny kernel.  A workgroup of those tiles walks all of K,
// so they win where K is short or their tiles are many, at every format of the
// scales.  N = 512 ... 7168, K = 1024 ... 8192, the weight out of memory / out of
// the last-level cache, split over workgroups against K groups, us:
// N = 4096: K = 2048, M = 32 -15 / -24 %, K = 4096 -6 / -18, K = 7168 +24 / -3,
// M = 64, K = 7168 +6 / -18; N = 2048, M = 64, K = 4096 -7 / -28, K = 5120 +19 /
// -15; N = 1024, K = 2048, M = 32 / 64 +7 / -11 out of memory, K = 4096 +40 / +17;
// N = 512, K = 7168 +87 / +58.  The line keeps every shape within 8 % of the
// better one out of memory, and gives up no gain there above 12 %.  Against the
// skinny kernel, M = 17 ... 32: N = 3600, K = 2048 +40 %, 4112 -2 ... -5, 7168 -6
// ... -20 (but K = 128 4.0 us / 4.6); from M = 33 -1 ... -56 % at every N and K.
SGL_RULE bool dense_k_groups(int64_t M, int64_t N, int64_t K, bool splits) {
  if (M > 64) return true;
  const int64_t tiles = (M + 31) / 32 * ((N + 63) / 64);
  return splits ? K <= 1024 || K <= 48 * tiles : M > 32 || (tiles >= 64 && K > 128);
}

// ---- grouped GEMMs of the MoE layer: 128-row tiles against the 32-row decode
// tiles, by the rows of an expert on average and the 128-row tiles there are
// when every expert has one.  The 32-row tiles stream each expert's weights
// once per tile (through L2); above 32 rows most experts fill a second one,
// while a 128-row tile takes the weights once.  But its tiles have to fill the
// CUs: over one or two rounds of them the last, partly filled round costs what
// the weights save.  From 64 rows the 128-row tiles always.
// Layer, 32-row / 128-row tiles in us, uniform and skewed load (`rounds`: tiles
// over CUs), bit-identical outputs:
//   FP8, 16 rounds (H = 4096, I = 2048, E = 256): 26 rows 1187 / 1249 and 1350 /
//     1287, 29 rows 1285 / 1256 and 1442 / 1291, 59 rows 1986 / 1364 and 2060 /
//     1465; 4 (E = 64): 29 rows 352 / 371 and 370 / 362, 36 rows 401 / 375 and 415 /
//     370; 2 (H = 2048, I = 1024, E = 64): 29 rows 114 / 140 and 130 / 138, 36 rows
//     135 / 143 and 135 / 140, 45 rows 157 / 146 and 157 / 143; 1 (E = 16): 29 rows
//     117 / 157 and 118 / 161, 45 rows 150 / 154 and 152 / 152, 58 rows 155 / 159
//     and 157 / 150; half a round (E = 8): 32 rows +6 and +8 %, 36 rows -29 and -26 %
//   FP4, 16: 29 rows 888 / 982 and 1008 / 1045, 38 rows 1142 / 1007 and 1134 /
//     1079; 4: 38 rows 346 / 306 and 324 / 340, 42 rows 350 / 305 and 349 / 342; 2
//     (E = 32): 46 rows -11 and +5 %, 52 rows -18 and -5 %; 1: 50 rows 138 / 112 and
//     139 / 154, 60 rows 169 / 122 and 169 / 157.
SGL_RULE bool moe_tall_tiles(bool fp4, int64_t rows, int64_t tiles, int64_t cus) {
  if (rows >= 64) return true;
  if (fp4) return (rows - 36) * tiles >= 28 * cus;
  return (rows - 29) * tiles >= 20 * cus || (rows > 32 && 2 * tiles <= cus);
}

// ---- MoE layer of the smallest batches: the two launches of moe_small.hip
// against the grouped path, where they fit (h in the workspace of the down
// projection's rows, and its quantized copy in the LDS of a CU) and are the
// faster.  Layer, grouped / these in us, E = 256 (64 within a few percent;
// tables with fragment copies 0 to 9 % more of the grouped path):
//   FP4, H = 4096, I = 2048: T k = 1 (T = 1) 81 / 18, 8 (T = 1) 74 / 41, 16 82 / 68,
//     24 (T = 3) 112 / 96, above which h leaves too little LDS for the weights;
//     H = 7168: 8 91 / 65, 24 (T = 3) 153 / 148.  Without a shared expert the
//     grouped path has two launches less: H = 4096, 12 53 / 49, 16 59 / 62; H =
//     7168, 8 68 / 58, 16 88 / 106; H = 5120, I = 1536, 16 71 / 70, 24 83 / 92.
//   FP8, whose grouped launches already are two and read at the memory's rate,
//     win by the launches saved only while the experts' bytes are few: H = 4096,
//     I = 2048, T = 1: k = 1 55 / 19, 8 64 / 57, 9 66 / 63, 12 76 / 79, 14 86 / 90;
//     H = 7168, k = 4 75 / 57, 5 78 / 65, 8 89 / 92; H = 3072, I = 1536, k = 16
//     62 / 66; H = 2048, I = 1024, k = 16 44 / 40.
//     T = 1 again where the grouped gate/up needs a second round of workgroups:
//     k = 16 at H = 4096 121 / 100, at 7168 167 / 162 (one round at H = 5120, I =
//     1536 93 / 111).
constexpr int kSmallMoeSlots = 64;  // T k: one lane a slot
constexpr int kSmallDownWaves = 16;
constexpr int kSmallDownLds = 157 * 1024;
// LDS of R = T (k + shared) rows: h as e4m3 with its scales, and the partial
// outputs of each line of K; the rest holds weights, 2 KB lines of each
// wavefront.
SGL_RULE int64_t small_down_rows_bytes(int64_t R, int64_t I) { return R * (I + I / 32 + I / 2); }
SGL_RULE int small_down_slots(int64_t R, int64_t I) {
  return (int)((kSmallDownLds - small_down_rows_bytes(R, I)) / (kSmallDownWaves * 2048));
}
SGL_RULE bool small_moe_ok(int64_t T, int64_t H, int64_t I, int k, int has_shared, bool fp4, int cus) {
  const int64_t S = T * k, R = T * (k + has_shared);
  if (S > (fp4 ? 24 : T > 1 ? 8 : kSmallMoeSlots)) return false;
  if (fp4 && !has_shared && S * H * I > (int64_t)16 * 5120 * 1536) return false;
  if (!fp4 && S * (H * I + (1 << 18)) > (int64_t)9 * (4096 * 2048 + (1 << 18)) &&
      !(T == 1 && (k + has_shared) * (I / 128) > cus))
    return false;
  return I <= H && small_down_rows_bytes(R, I) <= kSmallDownLds && small_down_slots(R, I) >= 2;
}

// ---- router projection, T > 256 tokens and H % 64 == 0: tokens x experts of a
// tile, and how its wavefronts share K.  The tiles are the largest that still
// give about a workgroup per CU, 64 x 128 as soon as 32 x 128 are more than one
// round of the 256 CUs (T = 6000, H = 4096, E = 256: 53 us in two rounds, 41 in
// one; but H = 1024, T = 4200 19.1 / 20.1, and three columns of tiles share x so
// well that the few tiles past a round fit beside it, one chain a workgroup, two
// workgroups a CU: T = 2752, E = 384, 258 tiles 35 / 39).  K over the four
// wavefronts (kSplit4, H % 128 == 0) for the 32 x 32 tiles (T = 512 13.0 -> 9.4
// us); for the larger ones over two or four groups of four wavefronts with a
// 64-deep K block each (kGroups), whose chain of stages is shorter.  What they
// save shows with x in the last-level cache, where the norm before the router
// has left it; with x out of memory (here: inputs past 256 MB in turn) the tiles
// wait for x, and some sizes lose a little.  E = 256, groups / without, x cached
// and x out of memory, us:
//   32 x 64 tiles: H = 2048, T = 3000 21.2 / 23.5 and 22.0 / 24.0; H = 4096, T = 2048
//     18.5 / 19.8 both, 3700 30.1 / 32.5 and 39.0 / 38.1; H = 7168, T = 3000 42.0 / 44.3
//     and 57.0 / 54.6; H = 4160, out of memory, T = 2048 19.0 / 23.7, 3000 37.8 / 35.5
//   32 x 128: H = 1024 18.3 / 18.0, 4096 28.5 / 29.7 and 32.7 / 33.2, 7168 39.9 / 43.0
//     and 47.8 / 48.8
//   64 x 128: H = 1024, T = 16384 out of memory 44.2 / 42.1; H = 2048, T = 12288 44.6 /
//     46.5 and 51.8 / 50.2; H = 4096, T = 6000 34.7 / 38.1 and 41.2 / 41.4, 8192 38.6 /
//     41.5 and 44.7 / 44.6, 16384 70.6 / 76.7 and 90.0 / 87.0; H = 7168, T = 8192 53.3 /
//     58.1 and 64.4 / 64.9; E = 128, H = 4096, T = 16384 39.6 / 40.8 and 53.8 / 51.4
// (A tile's K in one chain errs by 4.0e-7 of the logits, in two by 2.7e-7, in
// four by 1.9e-7, so no size goes to fewer chains than it had.)
enum RouterK { kOneChain, kSplit4, kGroups };
struct RouterTile {
  int tokens, experts;
  RouterK k;
};
SGL_RULE RouterTile router_tile(int64_t T, int64_t H, int64_t E) {
  const bool even = H % 128 == 0;
  const int64_t cols = (E + 127) / 128, rows = (T + 31) / 32;
  const int64_t t64 = rows * ((E + 63) / 64), t128 = rows * cols, tall = (T + 63) / 64 * cols;
  if (t128 > (cols >= 3 ? 264 : 256) && (H >= 2048 || tall >= 240))
    return {64, 128, H >= 2048 ? kGroups : kOneChain};
  if (t128 >= 240) return {32, 128, H >= 2048 && t128 <= 256 ? kGroups : kOneChain};
  if (t64 >= 240) return {32, 64, even || t64 <= 256 ? kGroups : kOneChain};
  return {32, 32, even ? kSplit4 : kOneChain};
}

// ---- permute (counting sort of the slots by expert): rounds of 1024 slots that
// one workgroup walks rather than chunks of them ranked and placed by many.  One
// workgroup / chunks with a table / without, us:
//   E = 256: 2048 slots 6.5 / 7.1 / 8.6, 2400 7.9 / 7.1 / 8.7, 3072 8.4 / 7.1 / 8.7,
//     4096 10.3 / 7.4 / 8.9, 15200 31.7 / 8.5 / 9.9, 65536 126 / 8.9 / 10.4
//   E = 32: 3072 7.1 / 6.7 / 8.4, 4096 8.5 / 6.8 / 8.4; E = 16: 2100 6.3 / 6.7 / 8.4, 3072
//     6.9 / 6.8 / 8.4, 3600 8.0 / 6.7 / 8.3, 4096 8.4 / 6.8 / 8.4; E = 1024: 2400 9.9 /
//     11.0 / 12.2
SGL_RULE int permute_rounds(int E, bool table) {
  return (table && E <= 512 ? 2 : 3) + (E <= (table ? 16 : 32) ? 1 : 0);
}

}  // namespace sgl
