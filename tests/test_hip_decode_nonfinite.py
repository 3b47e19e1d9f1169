"""Decode where scores are -inf, on the paths with fp32 weights (fp32 caches and
small pages), against the CPU oracle."""

from __future__ import annotations

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
