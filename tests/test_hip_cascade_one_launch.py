"""Cascade decode's two passes, in one launch or (long own tables of full batches) two: every pairing of their head tiles
(one tile or two, i.e. up to 16 or more query heads per workgroup), the edges of
blocks and splits on both sides, empty prefixes and empty own parts, and merges
of more partials than one round loads."""

from __future__ import annotations

import pytest
import torch

from kernel_lab.kv_cache import random_cascade_problem
from oracle import reference as ref
from tests.test_hip_cascade import check, expected, run

pytestmark = pytest.mark.gpu

OWN = [0, 1, 15, 16, 17, 63, 64, 65, 130, 257]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [32, 64, 128, 256])
@pytest.mark.parametrize(
    ("hq", "hkv", "batch"),
    [(8, 8, 2), (16, 4, 4), (16, 4, 10), (32, 1, 2), (20, 1, 10), (34, 2, 3)],
    ids=["tiles 1/1 one head", "1/1 full tile", "2/1", "2/2", "2/2 ragged groups", "2/2 two heads"],
)
def test_head_tiles(gpu_ops, dtype, head_dim, hq, hkv, batch):
    for prefix in (1, 257):
        q, c = random_cascade_problem(prefix, OWN[:batch], hq, hkv, head_dim, 16, dtype=dtype, device="cuda", seed=prefix + hq)
        check(run(gpu_ops, q, c), expected(q, c), dtype)


@pytest.mark.parametrize("head_dim", [64, 128])
def test_many_partials(gpu_ops, head_dim):
    """One unit: the prefix in 64 splits, the own tokens in up to 19."""
    q, c = random_cascade_problem(17000, [5000, 0, 300], 4, 1, head_dim, 16, dtype=torch.bfloat16, device="cuda")
    check(run(gpu_ops, q, c), expected(q, c), torch.bfloat16)


def test_no_prefix_pages(gpu_ops):
    q, c = random_cascade_problem(0, OWN, 32, 8, 128, 16, dtype=torch.float16, device="cuda")
    check(run(gpu_ops, q, c), expected(q, c), torch.float16)


@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("prefix", [0, 33, 300])
@pytest.mark.parametrize(("hq", "hkv"), [(64, 64), (192, 64), (1536, 64)], ids=["one head", "tiles 2/1", "2/2"])
def test_long_own_tables_of_full_batches(gpu_ops, head_dim, prefix, hq, hkv):
    """8 x 64 units pair, and tables of 4,096 tokens take a launch per pass; 4,080
    and less take one. The results of both match the oracle, empty rows too."""
    for longest in (4096, 4080):
        own = [longest, 0, 1, 16, 17, 65, 300, 129]
        if hq > 192:
            own[6] = 5
        q, c = random_cascade_problem(prefix, own, hq, hkv, head_dim, 16, dtype=torch.float16, device="cuda", seed=prefix + hq)
        check(run(gpu_ops, q, c), expected(q, c), torch.float16)


def test_grids_too_large_for_one_launch(gpu_ops):
    """2,050,000 sequences of 8 heads: 16.4 million workgroups for the own tokens and
    0.5 million for the prefix, together past 2^32 threads. Each takes a launch."""
    batch, at = 2_050_000, [0, 1_000_000, 2_033_599, 2_033_600, 2_049_999]
    g = torch.Generator(device="cuda").manual_seed(0)
    q = torch.randn(batch, 8, 32, generator=g, device="cuda").half()
    k, v = torch.randn(2, 2, 16, 8, 32, generator=g, device="cuda").half()
    table = torch.ones(batch, 1, dtype=torch.int32, device="cuda")
    lens = torch.full((batch,), 3, dtype=torch.int32, device="cuda")
    prefix = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.tensor([11], dtype=torch.int32, device="cuda")
    out = gpu_ops.cascade_decode_attention(q, k, v, *prefix, table, lens)
    assert (out != 0).any(-1).all()
    want = ref.cascade_decode_attention(q[at].cpu().float(), k.cpu(), v.cpu(), prefix[0].cpu(), prefix[1].cpu(), table[at].cpu(),
                                        lens[at].cpu())
    check(out[at], want, torch.float16)
