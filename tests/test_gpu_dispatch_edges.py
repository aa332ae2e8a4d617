"""Sizes on both sides of each dispatch rule, where a kernel choice changes:
the results against the oracle within the tolerances of the other layer tests."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_gemm_close, bf16_values, f32, to_dev_bf16, to_dev_f32
from oracle import moe as OM
from test_gpu_fp4 import fp4_table
from test_gpu_moe import table_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp4,T", [(False, 56), (False, 58), (True, 74), (True, 76)])
def test_moe_tile_rule(gpu, fp4, T):
    """Average rows per expert just below and at the 128-row tiles' threshold
    (FP8 29, FP4 38), with uneven groups (an expert with no row, one with one,
    the last with the rest)."""
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
