"""fp32 decode on the matrix cores, at the sizes where it can go wrong.

Lengths end inside, on and just past a 16-token block, a round of the
workgroup's waves (8 waves x 16 tokens; 4 x 16 where it runs four) and a page;
tails and spare pages hold NaN. Groups fill one head tile partly, wholly, and
two tiles (17 to 32 query heads per KV head) or several head groups. The oracle
is the float32 CPU path; decode_parity allows one fp32 ulp plus 1e-6.
"""

from __future__ import annotations

import pytest
import torch

from kernel_lab import _native
from kernel_lab.kv_cache import random_decode_problem
from oracle import reference as ref
from tests.conftest import decode_parity

pytestmark = pytest.mark.gpu

LENS = [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 257, 700]


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize(("hq", "hkv"), [(3, 3), (8, 2), (16, 1), (20, 1), (32, 1), (80, 2)])
@pytest.mark.parametrize("splits", [None, 1, 3])
def test_fp32_mfma_edges(gpu_ops, head_dim, hq, hkv, splits):
    page = 48 if splits == 3 else 16
    q, kv, _, _ = random_decode_problem(LENS, hq, hkv, head_dim, page, dtype=torch.float32, device="cuda",
                                        poison=float("nan"), tail=float("nan"), seed=head_dim + hq)
    out = gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens, num_splits=splits)
    want = ref.paged_decode_attention(q.cpu(), kv.k_cache.cpu(), kv.v_cache.cpu(), kv.block_table.cpu(), kv.seq_lens.cpu())
    decode_parity(out, want, torch.float32, f"{hq}/{hkv}/{head_dim} splits {splits}")


@pytest.mark.parametrize("head_dim", [64, 128, 256])
def test_fp32_mfma_is_no_further_from_64_bits_than_the_valu_kernel(gpu_ops, head_dim):
    """The scores and the block sums are added as trees, which keeps the result as
    near to 64 bits as the VALU kernel's short per-lane sums do; one running sum
    over head_dim 128 was twice as far. 2 % covers which inputs are drawn."""
    lens = [1 + (677 * b) % 4096 for b in range(15)] + [4096]
    q, kv, keys, values = random_decode_problem(lens, 32, 8, head_dim, 16, dtype=torch.float32, device="cuda")
    run = lambda: gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens).cpu().double()  # noqa: E731
    out = run()
    with _native.decode_switches(force_valu="1"):
        valu = run()
    want = torch.empty_like(out)
    for b in range(16):
        k = keys[b].cpu().double().transpose(0, 1)
        v = values[b].cpu().double().transpose(0, 1)
        w = torch.softmax(q[b].cpu().double().reshape(8, 4, head_dim) @ k.transpose(1, 2) * head_dim**-0.5, -1)
        want[b] = (w @ v).reshape(32, head_dim)
    errors = [((o - want).norm() / want.norm()).item() for o in (out, valu)]
    assert errors[0] <= 1.02 * errors[1], errors


def test_more_workgroups_than_eight_waves_allow(gpu_ops):
    """1,100,000 sequences of 8 KV heads, all but seven empty: a grid of 8.8 million
    workgroups, which 512 threads each would take past 2^32. Tables of 1,040 tokens,
    so the batch does not count as short."""
    batch, lens_at = 1_100_000, [0, 1, 500_000, 1_048_575, 1_048_576, 1_048_577, 1_099_999]
    g = torch.Generator(device="cuda").manual_seed(0)
    q = torch.randn(batch, 8, 64, generator=g, device="cuda")
    k, v = torch.randn(2, 1, 16, 8, 64, generator=g, device="cuda")
    table = torch.zeros(batch, 65, dtype=torch.int32, device="cuda")
    lens = torch.zeros(batch, dtype=torch.int32, device="cuda")
    lens[lens_at] = 5
    out = gpu_ops.paged_decode_attention(q, k, v, table, lens)
    assert int((out != 0).any(-1).any(-1).sum()) == len(lens_at)
    want = ref.paged_decode_attention(q[lens_at].cpu(), k.cpu(), v.cpu(), table[lens_at].cpu(), lens[lens_at].cpu())
    decode_parity(out[lens_at], want, torch.float32)
