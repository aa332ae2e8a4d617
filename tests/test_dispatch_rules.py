"""The size rules of the dispatches (csrc/sgl_rules.h), compiled for the host."""

from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "sglang-lite_amd" / "csrc"

WRAPPERS = r"""
#include "sgl_rules.h"
using namespace sgl;
extern "C" {
// the query of a workgroup of the attention grid (M, B, z), as its kernel names it
uint32_t attn_query(uint32_t x, uint32_t y, uint32_t M) { return y * M + attn_query_in_seq(x, M); }
uint32_t merge_groups(uint32_t queries, uint32_t heads) { return attn_merge_groups(queries, heads); }
void merge_at(uint32_t wg, uint32_t wave, uint32_t queries, uint32_t M, uint32_t heads, uint32_t* out) {
  const AttnMerge m = attn_merge_at(wg, wave, queries, M, heads);
  out[0] = m.query;
  out[1] = m.head;
}
int splits(int64_t queries, int heads, int64_t K, int cus) { return attn_plan(queries, heads, K, cus).nsplit; }
int few(int64_t queries, int heads, int64_t K, int cus) { return attn_plan(queries, heads, K, cus).few; }
int small_moe(int64_t T, int64_t H, int64_t I, int k, int shared, int fp4) {
  return small_moe_ok(T, H, I, k, shared, fp4, 256);
}
int router(int64_t T, int64_t H, int64_t E) {
  const RouterTile t = router_tile(T, H, E);
  return t.tokens * 10000 + t.experts * 10 + t.k;
}
int perm_rounds(int E, int table) { return permute_rounds(E, table); }
int tall(int fp4, int64_t rows, int64_t tiles, int64_t cus) { return moe_tall_tiles(fp4, rows, tiles, cus); }
int k_groups(int64_t M, int64_t N, int64_t K, int splits) { return dense_k_groups(M, N, K, splits); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.cpp", d / "rules.so"
    src.write_text(WRAPPERS)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-O1", "-shared", "-fPIC", f"-I{CSRC}",
                    str(src), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


@pytest.mark.parametrize("B,M", [(32, 1), (1, 8), (4, 8), (8, 4), (4, 2), (16, 3), (3, 16), (1, 24), (7, 1), (3, 3)])
@pytest.mark.parametrize("heads", [1, 6, 64, 70])
def test_attention_merge_covers_and_follows_the_splits(rules, B, M, heads):
    """Every (query, head) is merged once; with a multiple of eight queries by
    a workgroup of the XCD (linear workgroup index mod 8) of its splits."""
    Q = B * M
    ran_on = {rules.attn_query(x, y, M): (x + M * y) % 8 for y in range(B) for x in range(M)}
    assert sorted(ran_on) == list(range(Q))  # (split and head group z: x + M (y + B z), the same mod 8 if 8 | Q)
    seen = set()
    out = (ctypes.c_uint32 * 2)()
    for wg in range(rules.merge_groups(Q, heads)):
        for wave in range(4):
            rules.merge_at(wg, wave, Q, M, heads, out)
            q, h = out[0], out[1]
            if q >= Q or h >= heads:
                continue
            assert (q, h) not in seen
            seen.add((q, h))
            if Q % 8 == 0:
                assert ran_on[q] == wg % 8, f"query {q}"
    assert len(seen) == Q * heads


@pytest.mark.parametrize("cus", [256, 64, 1])
def test_attention_splits_fit_the_device(rules, cus):
    """At most a workgroup per CU once a query is split, none of them empty; the
    few-head kernel for at most 64 heads."""
    i64 = ctypes.c_int64
    for queries in (1, 7, 8, 32, 33, 100, 128, 129, 256, 5000):
        for heads in (1, 8, 64, 65, 128):
            for K in (0, 1, 64, 65, 192, 640, 2048, 100000):
                ns = rules.splits(i64(queries), heads, i64(K), cus)
                blocks = -(-K // 64)
                assert 1 <= ns <= 8
                assert heads <= 64 or not rules.few(i64(queries), heads, i64(K), cus)
                if ns > 1:
                    assert ns * queries * -(-heads // 64) <= cus
                    assert ns <= blocks and (ns - 1) * -(-blocks // ns) < blocks
    assert rules.splits(i64(32), 64, i64(640), 256) == 5
    assert rules.splits(i64(33), 64, i64(2048), 256) == 7


@pytest.mark.parametrize("queries,heads,K", [(33, 32, 256), (128, 16, 256), (128, 24, 384), (33, 32, 320),
                                             (128, 40, 512), (100, 1, 128)])
def test_attention_splits_only_where_the_merge_pays(rules, queries, heads, K):
    """Shapes whose merge costs more than the split saves, above all with bf16
    rows (33 queries x 32 heads x 256 indices: one split 14.0 us bf16, 17.7
    packed; four 16.7 and 17.3)."""
    assert rules.splits(ctypes.c_int64(queries), heads, ctypes.c_int64(K), 256) == 1


@pytest.mark.parametrize("queries,heads,K,few", [
    (1, 8, 64, 1), (1, 8, 256, 1), (32, 16, 256, 1), (16, 32, 192, 1), (1, 33, 64, 1), (256, 8, 128, 1),
    (1, 64, 640, 0), (32, 64, 640, 0), (256, 32, 640, 0), (2048, 64, 640, 0), (2048, 8, 640, 0), (1, 128, 64, 0),
    (1, 8, 1, 1), (1, 48, 1, 0), (64, 32, 32, 0), (64, 32, 33, 1),
])
def test_attention_kernel_by_chain(rules, queries, heads, K, few):
    """Short chains of few heads take the kernel that starts sooner."""
    assert rules.few(ctypes.c_int64(queries), heads, ctypes.c_int64(K), 256) == few


@pytest.mark.parametrize("M,N,K,splits,groups", [
    (17, 512, 3072, 1, 0), (32, 1024, 4096, 1, 0), (33, 1024, 7168, 1, 0), (32, 4096, 7168, 1, 0),
    (64, 1536, 8192, 1, 0), (32, 512, 1024, 1, 1), (32, 4096, 2048, 1, 1), (64, 4096, 4096, 1, 1),
    (17, 576, 7168, 0, 0), (32, 2112, 512, 0, 0), (33, 576, 7168, 0, 1), (32, 7168, 8192, 0, 1),
    (32, 4096, 128, 0, 0), (65, 512, 7168, 0, 1), (4096, 512, 7168, 0, 1),
])
def test_dense_k_groups_where_they_win(rules, M, N, K, splits, groups):
    """Long K over few tiles stays split over workgroups, narrow products of at
    most 32 rows on the skinny kernel."""
    i64 = ctypes.c_int64
    assert rules.k_groups(i64(M), i64(N), i64(K), splits) == groups


@pytest.mark.parametrize("fp4,rows,tiles,tall", [
    (0, 31, 4096, 1), (0, 29, 4096, 0), (0, 32, 1024, 0), (0, 36, 1024, 1), (0, 36, 512, 0), (0, 40, 512, 1),
    (0, 40, 256, 0), (0, 64, 256, 1), (0, 32, 128, 0), (0, 33, 128, 1), (0, 64, 1, 1),
    (1, 38, 4096, 1), (1, 37, 4096, 0), (1, 38, 1024, 0), (1, 43, 1024, 1), (1, 46, 512, 0), (1, 52, 512, 1),
    (1, 58, 256, 0), (1, 64, 256, 1),
])
def test_moe_tiles_need_rounds(rules, fp4, rows, tiles, tall):
    """128-row tiles below 64 rows an expert only where they fill the CUs often enough."""
    i64 = ctypes.c_int64
    assert rules.tall(fp4, i64(rows), i64(tiles), i64(256)) == tall


@pytest.mark.parametrize("fp4,T,H,I,k,small", [
    (0, 1, 3072, 1536, 12, 1), (0, 1, 3072, 1536, 16, 0), (0, 1, 7168, 2048, 5, 1),
    (0, 1, 4096, 2048, 8, 1), (0, 1, 4096, 2048, 9, 1), (0, 1, 4096, 2048, 12, 0), (0, 1, 4096, 2048, 14, 0),
    (0, 1, 4096, 2048, 16, 1), (0, 1, 7168, 2048, 4, 1), (0, 1, 7168, 2048, 8, 0), (0, 2, 7168, 2048, 4, 0),
    (0, 1, 7168, 2048, 16, 1), (0, 1, 5120, 1536, 12, 0), (0, 1, 5120, 1536, 16, 0), (0, 1, 2048, 1024, 16, 1),
    (0, 2, 4096, 2048, 4, 1), (0, 2, 512, 512, 5, 0), (0, 1, 256, 384, 2, 0),
    (1, 1, 4096, 2048, 16, 1), (1, 3, 4096, 2048, 8, 1), (1, 4, 4096, 2048, 8, 0), (1, 24, 4096, 2048, 1, 0),
])
def test_smallest_moe_batches_where_they_win(rules, fp4, T, H, I, k, small):
    """FP8 layers leave the two-launch path where their experts' bytes outweigh the launches."""
    i64 = ctypes.c_int64
    assert rules.small_moe(i64(T), i64(H), i64(I), k, 1, fp4) == small


@pytest.mark.parametrize("T,H,I,k,small", [(1, 4096, 2048, 8, 1), (1, 4096, 2048, 12, 1), (1, 4096, 2048, 16, 0),
                                           (2, 7168, 2048, 8, 0), (3, 5120, 1536, 8, 0), (3, 3072, 1536, 8, 1)])
def test_smallest_fp4_batches_without_a_shared_expert(rules, T, H, I, k, small):
    i64 = ctypes.c_int64
    assert rules.small_moe(i64(T), i64(H), i64(I), k, 0, 1) == small


@pytest.mark.parametrize("T,H,E,tile", [
    (512, 4096, 256, (32, 32, 1)), (512, 4160, 256, (32, 32, 0)), (2048, 4096, 256, (32, 64, 2)),
    (2048, 7168, 256, (32, 64, 2)), (3700, 4096, 256, (32, 64, 2)), (3000, 4160, 256, (32, 64, 0)),
    (2048, 4160, 256, (32, 64, 2)), (4096, 4096, 256, (32, 128, 2)), (4096, 1024, 256, (32, 128, 0)),
    (4097, 4096, 256, (64, 128, 2)), (4200, 1024, 256, (32, 128, 0)), (8192, 4096, 256, (64, 128, 2)),
    (8192, 1024, 256, (64, 128, 0)), (2752, 4096, 384, (32, 128, 0)), (2880, 4096, 384, (64, 128, 2)),
])
def test_router_tiles_where_they_win(rules, T, H, E, tile):
    """Tile and K split (0 one chain, 1 over four wavefronts, 2 groups) by both measured sides."""
    i64 = ctypes.c_int64
    got = rules.router(i64(T), i64(H), i64(E))
    assert (got // 10000, got % 10000 // 10, got % 10) == tile


@pytest.mark.parametrize("E,table,rounds", [(256, 1, 2), (256, 0, 3), (32, 1, 2), (32, 0, 4), (8, 1, 3), (1, 0, 4),
                                            (1024, 1, 3)])
def test_permute_chunks_where_they_win(rules, E, table, rounds):
    assert rules.perm_rounds(E, table) == rounds
