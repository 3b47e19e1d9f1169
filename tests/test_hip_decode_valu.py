"""The VALU decode kernel on the shapes that only it serves (head_dim 16; fp32 at
head_dim 32) and, by its switch, on those that the MFMA kernels take: page sizes on
and off the 16-token block, planned and given splits, NaN tails and spare pages,
empty sequences."""

from __future__ import annotations

import pytest
import torch

from kernel_lab import _native
from kernel_lab.kv_cache import random_decode_problem
from oracle import reference as ref
from tests.conftest import DTYPES, decode_parity

pytestmark = pytest.mark.gpu

LENS = [1, 4, 5, 15, 16, 17, 33, 63, 64, 65, 300, 1025, 9]


def _check(gpu_ops, hq, hkv, head_dim, page, dtype, splits):
    q, kv, _, _ = random_decode_problem(LENS, hq, hkv, head_dim, page, dtype=dtype, device="cuda", poison=float("nan"),
                                        tail=float("nan"), seed=page + hq)
    kv.seq_lens[-1] = 0
    out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits)
    want = ref.paged_decode_attention(q.cpu().float(), kv.k_cache.cpu(), kv.v_cache.cpu(), kv.block_table.cpu(), kv.seq_lens.cpu())
    decode_parity(out, want, dtype, f"{hq}/{hkv}/{head_dim} page {page} splits {splits}")


@pytest.mark.parametrize("page", [1, 5, 8, 16])
@pytest.mark.parametrize("splits", [None, 3, 64])
@pytest.mark.parametrize(
    ("dtype", "head_dim"), [(torch.float32, 16), (torch.float16, 16), (torch.bfloat16, 16), (torch.float32, 32)], ids=str
)
def test_shapes_of_its_own(gpu_ops, dtype, head_dim, page, splits):
    for hq, hkv in ((4, 4), (8, 2), (20, 1)):
        _check(gpu_ops, hq, hkv, head_dim, page, dtype, splits)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("page", [5, 8, 16])
@pytest.mark.parametrize(("hq", "hkv", "head_dim", "splits"), [(8, 2, 64, None), (32, 8, 128, 3), (6, 2, 256, None), (8, 1, 32, 7)])
def test_by_its_switch(gpu_ops, dtype, page, hq, hkv, head_dim, splits):
    with _native.decode_switches(force_valu="1"):
        _check(gpu_ops, hq, hkv, head_dim, page, dtype, splits)
