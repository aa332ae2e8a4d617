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

}  // namespace sgl
