"""FP8 decode on eight waves per unit (head_dim 128, launches of at most one
workgroup per CU) and on four (larger launches): lengths at the edges of a block,
of the waves' round (128 or 64 tokens) and of the segments a unit is cut into,
against the oracle's FP8 path."""

from __future__ import annotations

import pytest
import torch

from kernel_lab.kv_cache import quantize_fp8, random_decode_problem
from oracle import reference as ref
from tests.conftest import decode_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(("hq", "hkv"), [(32, 1), (20, 1), (16, 4), (8, 1), (5, 5)])
@pytest.mark.parametrize(
    "lens", [[1, 15, 16, 17, 127, 128, 129], [112, 113, 1023, 1025, 2500], [130] * 6, [0, 300, 0, 5000]], ids=str
)
def test_eight_wave_edges(gpu_ops, dtype, hq, hkv, lens):
    q, kv, _, _ = random_decode_problem([max(n, 1) for n in lens], hq, hkv, 128, 16, dtype=dtype, device="cuda",
                                        poison=float("nan"), seed=sum(lens) + hq)
    kv8, ks, vs = quantize_fp8(kv)
    kv8.seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out = gpu_ops.paged_decode_attention(q, kv8.k_cache, kv8.v_cache, kv8.block_table, kv8.seq_lens, k_scale=ks, v_scale=vs)
    keep = [b for b, n in enumerate(lens) if n]
    want = ref.paged_decode_attention_fp8(
        q[keep].cpu().float(), kv8.k_cache.cpu(), kv8.v_cache.cpu(), kv8.block_table[keep].cpu(), kv8.seq_lens[keep].cpu(),
        ks.cpu(), vs.cpu())
    decode_parity(out[keep], want, dtype, f"{hq}/{hkv} {lens}")
    assert all((out[b] == 0).all() for b, n in enumerate(lens) if n == 0)


@pytest.mark.parametrize("hq", [32, 8])
@pytest.mark.parametrize("batch", [256, 257])
def test_wave_count_changes_with_the_launch_size(gpu_ops, hq, batch):
    """One unit per sequence, and a table wide enough for the balanced schedule
    (4,096 tokens): 256 workgroups run eight waves, 257 four."""
    lens = [4096] + [[63, 64, 65, 127, 128, 129][b % 6] for b in range(batch - 1)]
    q, kv, _, _ = random_decode_problem(lens, hq, 1, 128, 16, dtype=torch.bfloat16, device="cuda", poison=float("nan"), seed=hq)
    kv8, ks, vs = quantize_fp8(kv)
    out = gpu_ops.paged_decode_attention(q, kv8.k_cache, kv8.v_cache, kv8.block_table, kv8.seq_lens, k_scale=ks, v_scale=vs)
    want = ref.paged_decode_attention_fp8(
        q.cpu().float(), kv8.k_cache.cpu(), kv8.v_cache.cpu(), kv8.block_table.cpu(), kv8.seq_lens.cpu(), ks.cpu(), vs.cpu())
    decode_parity(out, want, torch.bfloat16, f"{hq}/1 B={batch}")
