"""fp32 and small-page batches of short sequences, which run on the VALU kernel:
the sizes on either side of each line of the rule, against the oracle and against
the bits of the VALU kernel asked for by its switch."""

from __future__ import annotations

import pytest
import torch

from kernel_lab import _native
from kernel_lab.kv_cache import random_decode_problem
from oracle import reference as ref
from tests.conftest import decode_parity

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize(
    ("dtype", "page", "hq", "hkv", "head_dim", "batch", "longest", "valu"),
    [
        (F32, 16, 8, 8, 128, 4, 48, True),  # one head, a few blocks
        (F32, 16, 8, 8, 128, 4, 64, False),
        (F32, 16, 8, 8, 128, 64, 160, True),  # 512 units: up to 170 tokens x heads
        (F32, 16, 8, 8, 128, 64, 176, False),
        (F32, 16, 32, 8, 64, 96, 128, True),  # 4 heads: from 768 units
        (F32, 16, 32, 8, 64, 95, 128, False),
        (F32, 5, 64, 8, 256, 96, 30, True),
        (F32, 16, 72, 8, 256, 96, 16, False),  # 9 heads
        (BF16, 8, 8, 8, 64, 4, 128, True),
        (BF16, 8, 8, 8, 64, 4, 136, False),
        (F16, 8, 16, 8, 64, 64, 384, True),  # 512 units: up to 768
        (F16, 8, 16, 8, 64, 64, 392, False),
        (BF16, 1, 8, 8, 128, 96, 192, True),  # 768 units: up to 192
        (BF16, 1, 8, 8, 128, 96, 193, False),
        (F16, 12, 4, 2, 32, 256, 300, True),
        (F16, 12, 12, 4, 32, 256, 24, False),  # 3 heads
        (BF16, 8, 32, 8, 256, 96, 64, True),
        (BF16, 8, 32, 8, 256, 96, 72, False),
    ],
)
def test_either_side_of_the_line(gpu_ops, dtype, page, hq, hkv, head_dim, batch, longest, valu):
    lens = [longest] + [1 + (7 * b) % longest for b in range(1, batch)]
    q, kv, _, _ = random_decode_problem(lens, hq, hkv, head_dim, page, dtype=dtype, device="cuda", poison=float("nan"),
                                        tail=float("nan"), seed=batch + longest)
    kv.seq_lens[2] = 0
    run = lambda: gpu_ops.paged_decode_attention(q, kv.k_cache, kv.v_cache, kv.block_table, kv.seq_lens).cpu()  # noqa: E731
    out = run()
    with _native.decode_switches(force_valu="1"):
        forced = run()
    if valu:
        assert torch.equal(out, forced)
    elif dtype == F32:
        assert not torch.equal(out, forced)  # the two kernels round differently
    want = ref.paged_decode_attention(q.cpu().float(), kv.k_cache.cpu(), kv.v_cache.cpu(), kv.block_table.cpu(), kv.seq_lens.cpu())
    decode_parity(out, want, dtype, f"{hq}/{hkv}/{head_dim} B={batch} T={longest}")
    decode_parity(forced, want, dtype, "VALU")
