"""Decode at the edges of the number range, on the paths with fp32 weights (fp32
caches and small pages): scores of -inf against the CPU oracle, and weights
below the normal range."""

from __future__ import annotations

import math

import pytest
import torch

from kernel_lab.kv_cache import random_decode_problem
from oracle import reference as ref
from tests.conftest import decode_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("dtype", "page"), [(torch.float32, 16), (torch.float32, 8), (torch.float16, 8), (torch.bfloat16, 5)])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("masked", [(16, 128), (1, 700), (0, 16), (690, 700)], ids=str)
def test_blocks_of_minus_infinity(gpu_ops, dtype, page, splits, masked):
    """Tokens that score -inf weigh nothing, also where a wave's first block or
    a whole split holds no others."""
    q, kv, _, _ = random_decode_problem([700, 40], 8, 2, 128, page, dtype=dtype, device="cuda")
    q[..., 3] = q[..., 3].abs() + 0.5
    for tok in range(*masked):
        kv.k_cache[int(kv.block_table[0, tok // page]), tok % page, :, 3] = -float("inf")
    out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits)
    want = ref.paged_decode_attention(q.cpu().float(), kv.k_cache.cpu(), kv.v_cache.cpu(), kv.block_table.cpu(), kv.seq_lens.cpu())
    decode_parity(out, want, dtype, f"{masked}")


@pytest.mark.parametrize("page", [16, 8])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("far", [17, 255])
def test_weights_below_the_normal_range(gpu_ops, page, splits, far):
    """One value of 1e38 at a weight of e^-90 (2^-130, a subnormal: 19 bits)
    among zeros. 1e-4 covers the subnormal's rounding (2^-20), its split's
    normaliser and the exponent's (90 / ln 2 at 2^-24 of itself)."""
    q, kv, _, _ = random_decode_problem([256], 4, 1, 64, page, dtype=torch.float32, device="cuda")
    q.zero_()
    q[..., 0] = 8.0
    kv.k_cache.zero_()
    kv.v_cache.zero_()
    kv.k_cache[..., 0] = 90.0
    at = (int(kv.block_table[0, far // page]), far % page, 0)
    kv.k_cache[at][0] = 0.0
    kv.v_cache[at] = 1e38
    out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits)
    want = math.exp(-90.0) / 255 * 1e38
    assert (out.cpu().double() - want).abs().max() <= 1e-4 * want
