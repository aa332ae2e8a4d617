"""Sizes on both sides of each dispatch rule, where a kernel choice changes:
the results against the oracle within the tolerances of the other layer tests."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_gemm_close, assert_layer_close, bf16_values, f32, to_dev_bf16, to_dev_f32
from oracle import attn as OA
from oracle import kv as OK
from oracle import moe as OM
from test_gpu_fp4 import fp4_table
from test_gpu_moe import table_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp4,T", [(False, 56), (False, 58), (True, 74), (True, 76), (False, 64), (False, 66),
                                   (True, 126), (True, 128)])
def test_moe_tile_rule(gpu, fp4, T):
    """Average rows per expert just below and at the 128-row tiles' threshold
    (with these few tiles FP8 33, FP4 64), with uneven groups (an expert with
    no row, one with one, the last with the rest)."""
    from sglang_lite_amd import moe as M

    rng = np.random.default_rng(T + fp4)
    H, I, E, k = 512, 512, 4, 2
    print(f"tile rule fp4={fp4} T={T} rows/expert={T * k // E}", flush=True)
    ids = np.tile(np.array([[3, 2]], np.int32), (T, 1))
    ids[0, 1] = 1
    x = bf16_values(rng, (T, H))
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    make = OM.make_fp4_expert if fp4 else OM.make_expert
    experts = [make(rng, H, I) for _ in range(E)]
    sh = OM.make_expert(rng, H, I)
    table = (fp4_table if fp4 else table_from)(experts, sh, gpu)
    y = M.moe_forward(to_dev_bf16(x, gpu), torch.from_numpy(ids).to(gpu), to_dev_f32(w, gpu), table)
    assert_gemm_close(f32(y), OM.moe_forward(x, ids, w, experts, sh), f"tile rule T={T}")


@pytest.mark.parametrize("fp4,T,H,I,E,k,shared,mode", [
    (False, 1, 4096, 2048, 12, 8, True, 0),
    (False, 1, 4224, 384, 20, 16, False, 2),   # 33 K lines, 16 slots, no shared expert
    (False, 2, 512, 512, 4, 4, True, 3),       # 8 slots; power-of-two scales
    (False, 2, 640, 512, 6, 5, True, 0),       # 10 slots: the grouped path
    (False, 1, 256, 384, 4, 2, True, 0),       # I > H: the grouped path
    (True, 1, 4096, 2048, 10, 8, True, 3),
    (True, 1, 512, 256, 3, 1, True, 0),        # fewer K lines than wavefronts
    (True, 3, 2560, 2304, 9, 8, True, 1),      # 24 slots, I past 16 lines
    (True, 4, 512, 512, 7, 6, False, 2),       # 24 slots, no shared expert
    (True, 12, 512, 512, 5, 2, True, 3),       # 24 slots, rows of the shared expert 12
    (True, 24, 512, 512, 5, 1, True, 0),       # two 16-row tiles of the shared expert
    (True, 5, 512, 512, 7, 5, True, 3),        # 25 slots: the grouped path
])
def test_moe_smallest_batches(gpu, fp4, T, H, I, E, k, shared, mode):
    """The layer of one to a few tokens and the sizes where it gives way to
    the grouped path; an id outside the experts adds nothing, and a token may
    name an expert twice (the oracle: the same slot with weight 0, and a copy
    of that expert under an id of its own)."""
    from sglang_lite_amd import moe as M

    rng = np.random.default_rng(T * 1000 + H + I + mode)
    print(f"smallest fp4={fp4} T={T} H={H} I={I} E={E} k={k} shared={shared} mode={mode}", flush=True)
    x = bf16_values(rng, (T, H))
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    dev_ids, ref_w = ids.copy(), w.copy()
    if T * k > 8:
        dev_ids[0, k - 1], ref_w[0, k - 1] = (-1 if T % 2 else E), 0.0
    if k > 2:
        dev_ids[T - 1, 1], ids[T - 1, 1] = ids[T - 1, 0], E
    ue = mode in (1, 3)
    experts = [OM.make_fp4_expert(rng, H, I) if fp4 else OM.make_expert(rng, H, I, ue8m0=ue) for _ in range(E)]
    sh = OM.make_expert(rng, H, I, ue8m0=ue) if shared else None
    table = (fp4_table if fp4 else table_from)(experts, sh, gpu)
    y = M.moe_forward(to_dev_bf16(x, gpu), torch.from_numpy(dev_ids).to(gpu), to_dev_f32(w, gpu), table,
                      swiglu_limit=3.0, scale_mode=mode)
    experts = experts + [experts[ids[T - 1, 0]]]
    y_ref = OM.moe_forward(x, ids, ref_w, experts, sh, swiglu_limit=3.0, mode=mode)
    assert_layer_close(f32(y), y_ref, f"smallest T={T} k={k}")


@pytest.mark.parametrize("scales", ["fp32", "e8m0", "mixed"])
@pytest.mark.parametrize("M,N,K", [
    (17, 208, 128),     # one K block (three of a stage's four groups idle), a ragged column tile
    (33, 1040, 640),    # five K blocks: a last stage of one
    (64, 1600, 256),    # split-K shape that the K groups take; two K blocks
    (32, 512, 4096),    # split-K shape that stays split
    (130, 2048, 896),   # 5 x 32 tiles of 32 x 64, seven K blocks
    (257, 2048, 384),   # past one round of 32 x 64: 32 x 128, an odd K block at the end
    (513, 2048, 7168),  # past one round of 32 x 128: 64 x 128, the longest K its scale table holds
    (500, 2048, 7296),  # one K block more: the tiles before
    (200, 512, 8192),   # the longest K of the 32-row tiles' scale table
    (200, 512, 8320),
    (2060, 1536, 256),  # few 256 x 256 tiles: several rounds of 64 x 128
])
def test_fp8_gemm_k_groups(gpu, M, N, K, scales):
    """The dense product on both sides of each tile rule against the
    dequantized product, in both output types."""
    from sglang_lite_amd import kernel as KK
    from sglang_lite_amd import v4_deep_gemm as DG

    print(f"k groups M={M} N={N} K={K} {scales}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=gen, device=gpu).bfloat16()
    b = (torch.randn(N, K, generator=gen, device=gpu) * 90).clamp_(-448, 448).to(torch.float8_e4m3fn)
    nb = (N + 127) // 128
    if scales == "fp32":
        a, sa = KK.act_quant(x, 128)
        sb = torch.rand(nb, K // 128, generator=gen, device=gpu) * 1e-4 + 1e-4
    else:
        a, sa = KK.act_quant(x, 128, "ue8m0", torch.float8_e8m0fnu)
        sb = torch.randint(110, 118, (nb, K // 128), generator=gen, device=gpu, dtype=torch.uint8).view(
            torch.float8_e8m0fnu)
        if scales == "mixed":
            sb = sb.float()
    ad = a.double() * sa.float().double().repeat_interleave(128, 1)
    bd = b.double() * sb.float().double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)
    ref = (ad @ bd.t().contiguous()).float().cpu().numpy()
    for dt in (torch.bfloat16, torch.float32):
        c = DG.fp8_gemm_nt(a, sa, b, sb, out_dtype=dt)
        assert c.dtype == dt
        assert_gemm_close(f32(c) if dt == torch.bfloat16 else c.cpu().numpy(), ref, f"{M}x{N}x{K} {scales} {dt}")


def _attn(gpu, q, kv, sink, idx, scale, fmt):
    """(device output, the rows as the device reads them) for a bf16 cache,
    packed rows or packed pages of 3 rows (not a power of two)."""
    from sglang_lite_amd import dsv4_kv_pack as KVP
    from sglang_lite_amd import v4_sparse_mla as SA

    qd, kvd, sd = to_dev_bf16(q, gpu), to_dev_bf16(kv, gpu), to_dev_f32(sink, gpu)
    idd = torch.from_numpy(idx).to(gpu)
    if fmt == "bf16":
        return f32(SA.sparse_attn(qd, kvd, sd, idd, scale)), kv
    packed = KVP.pack_dsv4_kv_bf16(kvd)
    rows = np.stack([OK.dequant_row_a(p.cpu().numpy()) for p in packed])
    cache = packed if fmt == "rows" else torch.stack([KVP.to_paged_hnd(p, 3) for p in packed])
    return f32(SA.sparse_attn_packed(qd, cache, sd, idd, scale, n_rows=kv.shape[1])), rows


@pytest.mark.parametrize("fmt", ["bf16", "rows", "pages"])
@pytest.mark.parametrize("H", [1, 8, 32, 33, 64, 100])
def test_sparse_attn_row_counts_at_block_edges(gpu, H, fmt):
    """Valid rows per query at the edges of the 32-row blocks and of the tile
    ring, masked entries between them, head counts at the edges of the
    16- and 32-head tiles and of the 64-head groups."""
    counts = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 130]
    rng = np.random.default_rng(H)
    S, n, K = len(counts), 150, 160
    print(f"attn edges H={H} {fmt}", flush=True)
    q, kv = bf16_values(rng, (1, S, H, 512)), bf16_values(rng, (1, n, 512))
    sink = (rng.standard_normal(H) * 2).astype(np.float32)
    idx = np.full((1, S, K), -1, np.int32)
    for s, c in enumerate(counts):
        idx[0, s, np.sort(rng.permutation(K)[:c])] = rng.permutation(n)[:c]
    got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, fmt)
    assert_gemm_close(got, OA.sparse_attn_blocked(q, rows, sink, idx, 512 ** -0.5), f"H={H} {fmt}")
    assert np.all(got[0, 0] == 0)


@pytest.mark.parametrize("fmt,K", [("bf16", 2752), ("bf16", 2753), ("rows", 1792), ("pages", 1793)])
@pytest.mark.parametrize("queries", [1, 300])
def test_sparse_attn_row_list_edges(gpu, fmt, K, queries):
    """As many indices as the row list of a workgroup holds rows, and one more,
    every seventh masked (300 queries: unsplit; one: split, a list each; lists
    filled exactly and past their end by valid rows:
    test_sparse_attn_row_lists_by_valid_rows)."""
    rng = np.random.default_rng(K)
    print(f"attn list K={K} queries={queries} {fmt}", flush=True)
    q, kv = bf16_values(rng, (1, queries, 2, 512)), bf16_values(rng, (1, 40, 512))
    sink = rng.standard_normal(2).astype(np.float32)
    idx = rng.integers(0, 40, (1, queries, K)).astype(np.int32)
    idx[0, :, ::7] = -1
    got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, fmt)
    for s in (0, queries - 1):  # each query by itself: the oracle gathers every row
        ref = OA.sparse_attn_exact(q[:, s:s + 1], rows, sink, idx[:, s:s + 1], 512 ** -0.5)
        assert_gemm_close(got[:, s:s + 1], ref, f"K={K} query {s}")


@pytest.mark.parametrize("queries", [8, 9, 24])
@pytest.mark.parametrize("H", [6, 64, 70])
def test_sparse_attn_merge_order(gpu, queries, H):
    """The values of split rows merged in both orders of workgroups (a multiple
    of eight queries or not), head counts that do not fill a workgroup's four
    (where each merge runs: test_dispatch_rules.py)."""
    rng = np.random.default_rng(queries + H)
    K = 1024
    print(f"attn merge H={H} queries={queries}", flush=True)
    q, kv = bf16_values(rng, (1, queries, H, 512)), bf16_values(rng, (1, 60, 512))
    sink = rng.standard_normal(H).astype(np.float32)
    idx = rng.integers(0, 60, (1, queries, K)).astype(np.int32)
    got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, "bf16")
    assert_gemm_close(got, OA.sparse_attn_blocked(q, rows, sink, idx, 512 ** -0.5), f"H={H} queries={queries}")


@pytest.mark.parametrize("order", ["rising", "falling", "one late"])
def test_sparse_attn_moving_reference(gpu, order):
    """Scores that rise block after block (the reference moves in each), fall,
    or jump in the last block; and a row 0 that no query selects holding
    infinities and NaN (the rows that pad a block read zeros, never it)."""
    rng = np.random.default_rng(len(order))
    n, K, H, S = 201, 200, 64, 260
    q = np.zeros((1, S, H, 512), np.float32)
    q[..., 0] = 8.0
    q[..., 1:4] = bf16_values(rng, (1, S, H, 3))
    kv = bf16_values(rng, (1, n, 512))
    rank = {"rising": np.arange(K), "falling": np.arange(K)[::-1], "one late": (np.arange(K) == 199) * 150}
    kv[0, 1:, 0] = np.float32(0.25) * np.floor(rank[order] * 0.5)  # scores up to 200 apart, exact in bf16
    kv[0, 0] = np.array([np.inf, np.nan] * 256, np.float32)
    idx = np.broadcast_to(np.arange(1, n, dtype=np.int32), (1, S, K)).copy()
    sink = rng.standard_normal(H).astype(np.float32)
    got, _ = _attn(gpu, q, kv, sink, idx, 1.0, "bf16")
    ref = OA.sparse_attn_exact(q[:, :1], kv, sink, idx[:, :1], 1.0)
    assert np.all(np.isfinite(got))
    assert_gemm_close(got[:, :1], ref, order)
    for s in (1, S - 1):
        assert_gemm_close(got[:, s:s + 1], OA.sparse_attn_exact(q[:, s:s + 1], kv, sink, idx[:, s:s + 1], 1.0), order)


@pytest.mark.parametrize("T,H,E", [
    (4096, 448, 256),   # 32 x 128 tiles in exactly one round; 7 K blocks for two groups
    (4097, 64, 256),    # 64 x 128 tiles, one row past that round; the second group has no K block
    (4110, 192, 250),   # ragged last tiles of both sides, 3 K blocks
    (1921, 320, 256),   # 32 x 64 tiles, 5 K blocks for four groups
    (2049, 64, 248),    # 32 x 64 tiles, one K block: three groups have none
    (1920, 384, 256),   # 32 x 64 tiles from here (240), 6 K blocks
    (2049, 192, 256),   # an odd number of K blocks in two rounds: one chain
    (4096, 2048, 256),  # 32 x 128 tiles, two groups
    (4097, 2112, 250),  # 64 x 128 tiles, two groups, 33 K blocks
    (7680, 256, 256),   # 64 x 128 tiles of short rows: one chain
    (7679, 256, 250),   # ... 32 x 128 below 240 of them
    (2752, 256, 320),   # three columns of 32 x 128 tiles a little past one round
    (1919, 384, 192),   # the four-way split's 32 x 32 tiles
])
def test_router_k_groups(gpu, T, H, E):
    """The projection at the edges of its tile rule and with K blocks that the
    groups share unevenly, within the fp32 summation bound of the exact logits:
    H products summed in at most H additions of partial sums no larger than the
    sum of magnitudes, in practice well below 2^-21 of it."""
    from sglang_lite_amd import moe as M

    print(f"router k groups T={T} H={H} E={E}", flush=True)
    rng = np.random.default_rng(T + H + E)
    x = bf16_values(rng, (T, H))
    W = bf16_values(rng, (E, H))
    lg = torch.full((T, E), float("nan"), dtype=torch.float32, device=gpu)
    M.gate(to_dev_bf16(x, gpu), to_dev_bf16(W, gpu), 4, "sigmoid", None, 1.0, logits=lg)
    exact = x.astype(np.float64) @ W.astype(np.float64).T
    mag = np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64).T
    assert np.all(np.abs(f32(lg).astype(np.float64) - exact) <= 2.0 ** -21 * mag + 1e-30)


@pytest.mark.parametrize("T,k,E", [
    (384, 8, 256),    # 3072 slots: the largest of one workgroup
    (439, 7, 256),    # 3073: four chunks, one slot in the last
    (700, 6, 1024),   # chunks doubled so that their table fits in the slots, no idle expert thread
    (5000, 1, 1),     # one expert: every thread sums a part of the table
    (4096, 1, 1),     # ... and the four rounds of one workgroup before
    (70001, 1, 1),    # ... 69 chunks: more parts than chunks have
    (140000, 1, 3),   # 341 parts, halved with an odd one left over
    (40000, 2, 100),  # ten parts: one halving
    (2048, 2, 8),     # eight experts: four rounds of one workgroup
    (2049, 2, 8),     # ... and chunks
    (2001, 3, 1000),  # experts that do not divide the workgroup's threads
    (16385, 8, 200),  # chunks of two rounds
])
def test_permute_chunks(gpu, T, k, E):
    """The chunked counting sort at its size edges, bit for bit."""
    from sglang_lite_amd import moe as M

    print(f"permute chunks T={T} k={k} E={E}", flush=True)
    rng = np.random.default_rng(T + k + E)
    ids = np.argsort(rng.standard_normal((T, E)) + np.linspace(0, 2, E), axis=1)[:, :k].astype(np.int32)
    ref = OM.permute(ids, E)
    for got, name in zip(M.permute(torch.from_numpy(ids).to(gpu), E),
                         ("counts", "offsets", "sorted_slot", "slot_pos")):
        np.testing.assert_array_equal(got.cpu().numpy(), ref[name], err_msg=name)


@pytest.mark.parametrize("T", [128, 129, 300])
def test_layer_permute_rounds(gpu, T):
    """The layer on both sides of the chunked sort's threshold (2048 slots),
    with the table in its workspace."""
    from sglang_lite_amd import moe as M

    print(f"layer permute T={T}", flush=True)
    rng = np.random.default_rng(T)
    H, I, E, k = 256, 256, 20, 16
    ids = np.argsort(rng.standard_normal((T, E)), axis=1)[:, :k].astype(np.int32)
    x = bf16_values(rng, (T, H))
    w = rng.uniform(0.1, 1.0, (T, k)).astype(np.float32)
    experts = [OM.make_expert(rng, H, I) for _ in range(E)]
    sh = OM.make_expert(rng, H, I)
    y = M.moe_forward(to_dev_bf16(x, gpu), torch.from_numpy(ids).to(gpu), to_dev_f32(w, gpu),
                      table_from(experts, sh, gpu))
    assert_gemm_close(f32(y), OM.moe_forward(x, ids, w, experts, sh), f"layer permute T={T}")


@pytest.mark.parametrize("queries,H,K", [(8, 64, 192), (16, 64, 256), (32, 64, 384), (33, 64, 384), (32, 8, 256),
                                         (64, 16, 384), (33, 100, 640), (300, 64, 200),
                                         (300, 2, 2000), (257, 33, 3600), (1, 64, 20000)])  # lists of several parts
def test_sparse_attn_formats_split_alike(gpu, queries, H, K):
    """Packed rows and pages give bit for bit what their dequantized rows give,
    at sizes where one split or several are close."""
    rng = np.random.default_rng(queries + H + K)
    print(f"attn formats queries={queries} H={H} K={K}", flush=True)
    n = 96
    q, kv = bf16_values(rng, (1, queries, H, 512)), bf16_values(rng, (1, n, 512))
    sink = rng.standard_normal(H).astype(np.float32)
    idx = rng.integers(-1, n, (1, queries, K)).astype(np.int32)
    got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, "rows")
    paged, _ = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, "pages")
    plain, _ = _attn(gpu, q, rows, sink, idx, 512 ** -0.5, "bf16")
    np.testing.assert_array_equal(got, plain)
    np.testing.assert_array_equal(paged, plain)


@pytest.mark.parametrize("valid", [1727, 1728, 1729, 1792, 1793, 2688, 2752, 2753, 3600])
@pytest.mark.parametrize("K", [3600, 5000])
def test_sparse_attn_row_lists_by_valid_rows(gpu, valid, K):
    """Valid rows that fill the list (1792 packed, 2752 bf16) or pass it, between
    masked entries: the formats bit for bit, and the exact softmax."""
    rng = np.random.default_rng(valid + K)
    print(f"attn lists valid={valid} K={K}", flush=True)
    S, H, n = 257, 2, 64
    q, kv = bf16_values(rng, (1, S, H, 512)), bf16_values(rng, (1, n, 512))
    sink = rng.standard_normal(H).astype(np.float32)
    idx = np.full((1, S, K), -1, np.int32)
    for s in range(S):
        idx[0, s, np.sort(rng.permutation(K)[:valid])] = rng.integers(0, n, valid)
    got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, "rows")
    plain, _ = _attn(gpu, q, rows, sink, idx, 512 ** -0.5, "bf16")
    np.testing.assert_array_equal(got, plain)
    for s in (0, S - 1):
        ref = OA.sparse_attn_exact(q[:, s:s + 1], rows, sink, idx[:, s:s + 1], 512 ** -0.5)
        assert_gemm_close(got[:, s:s + 1], ref, f"valid={valid} query {s}")


@pytest.mark.parametrize("fmt", ["bf16", "rows", "pages"])
@pytest.mark.parametrize("H,K", [(1, 1), (8, 63), (8, 64), (8, 65), (8, 256), (16, 300), (31, 128), (32, 130),
                                 (33, 64), (40, 100), (63, 64), (64, 1)])
def test_sparse_attn_short_chains(gpu, H, K, fmt):
    """The kernel of few heads and short selections (one to a few blocks, split
    or not, both sides of its 32 heads), masked entries among the rows, a query
    with none."""
    rng = np.random.default_rng(H * 1000 + K)
    print(f"attn short H={H} K={K} {fmt}", flush=True)
    for B, S in ((1, 2), (3, 1), (2, 64)):
        n = 70
        q, kv = bf16_values(rng, (B, S, H, 512)), bf16_values(rng, (B, n, 512))
        sink = (rng.standard_normal(H) * 2).astype(np.float32)
        idx = rng.integers(0, n, (B, S, K)).astype(np.int32)
        idx[rng.random(idx.shape) < 0.2] = -1
        idx[0, 0] = -1
        got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, fmt)
        assert_gemm_close(got, OA.sparse_attn_blocked(q, rows, sink, idx, 512 ** -0.5), f"H={H} K={K} {fmt} {B}x{S}")
        assert np.all(got[0, 0] == 0)


@pytest.mark.parametrize("fmt", ["bf16", "pages"])
@pytest.mark.parametrize("H,K", [(8, 64), (8, 130), (16, 192), (8, 640), (40, 64)])
def test_sparse_attn_few_heads_masked_blocks(gpu, H, K, fmt):
    """The kernel of few heads where whole blocks of 64 indices are masked: at
    the end (left out), at the head, between others, everywhere."""
    rng = np.random.default_rng(H + K)
    print(f"attn masked blocks H={H} K={K} {fmt}", flush=True)
    n, S = 90, 9
    q, kv = bf16_values(rng, (1, S, H, 512)), bf16_values(rng, (1, n, 512))
    sink = rng.standard_normal(H).astype(np.float32)
    idx = rng.integers(0, n, (1, S, K)).astype(np.int32)
    for s, keep in enumerate((0, 1, 63, 64, 65, K - 1, K)):  # a prefix of valid entries
        idx[0, s, keep:] = -1
    idx[0, 7, :K - 1] = -1
    idx[0, 8, 1:K - 1] = -1
    got, rows = _attn(gpu, q, kv, sink, idx, 512 ** -0.5, fmt)
    assert_gemm_close(got, OA.sparse_attn_blocked(q, rows, sink, idx, 512 ** -0.5), f"H={H} K={K} {fmt}")
    assert np.all(got[0, 0] == 0)
